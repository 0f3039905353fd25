"""The f32 Jeff kernel at hd 256 on bf16 planes (grids above two workgroups per
CU) where its tiling can go wrong: 4, 2 and 1 query heads per workgroup, lengths
and key spans that end inside a 32-key tile, lengths that are no multiple of 4,
a head dim below the padded one, RoPE widths inside and outside the in-register
path, trimmed rows, and value tiles whose magnitudes jump by far more than a
half-precision number's range. Against the oracle; an output is a
convex combination of its head's values up to its position times a gate, so
the tolerance is 2e-5 (the f32 one at order 1) of the largest such value
(test_jeff_ranges weighs each value by its probability). And scores and values
that are inf or NaN, kept and masked: the oracle's pattern, finite outputs within 2e-5.
"""
import numpy as np
import pytest

import oracle
import tenferro_ext as te
from tenferro_ext.workloads import Lcg


@pytest.mark.gpu
@pytest.mark.parametrize("rows,L,heads,kv,hd,rot,trim,jumps", [
    (5, 333, 8, 2, 256, 64, True, True), (9, 250, 4, 2, 256, 64, False, True),
    (6, 481, 3, 3, 256, 32, False, False), (7, 289, 6, 2, 200, 50, True, False),
    (17, 97, 8, 2, 256, 0, False, True)])
def test_split_rows_gpu(gpu_ctx, rows, L, heads, kv, hd, rot, trim, jumps):
    print(f"[split] {rows} x {L}, heads {heads}/{kv} x {hd}, rot {rot}, trim {trim}", flush=True)
    rng = Lcg(rows * 1000 + L)
    q, gate = (rng.normal(rows * heads * hd * L).astype(np.float32) for _ in range(2))
    k, v = (rng.normal(rows * kv * hd * L).astype(np.float32) for _ in range(2))
    v = v.reshape(rows, kv * hd, L)
    if jumps:
        for t, e in enumerate((0, -20, 12, 40, -40, 3, 0, 90, -90, 1, 0)):
            v[:, :, 32 * t:32 * t + 32] *= np.float32(2.0 ** e)
    qn, kn = ((rng.normal(hd) * 0.1).astype(np.float32) for _ in range(2))
    mask = np.ones((rows, L), np.float32)
    for r in range(rows):
        mask[r, :(37 * r) % (L - 3)] = 0.0   # left padding
        mask[r, -(r % 4) or L:] = 0.0        # and inactive last keys
        mask[r, L // 2] = 0.0
    args = (q, k, v.reshape(-1), gate, qn, kn, mask.reshape(-1), rows, L, heads, kv, hd, rot,
            1.0e7, 1.0e-6)
    oracle.set_threads(8)
    want = oracle.jeff_rows(*args, trim_leading=trim).reshape(rows, heads, hd, L)
    got = np.asarray(te.jeff_full_attention_rows(*args, trim_leading=trim, ctx=gpu_ctx))
    got = got.reshape(rows, heads, hd, L)
    big = np.maximum.accumulate(np.abs(v * mask[:, None, :]).reshape(rows, kv, hd, L).max(2), axis=-1)
    big = np.repeat(big, heads // kv, axis=1)[:, :, None, :]
    assert np.isfinite(got).all()
    err = np.abs(got - want)
    assert (err <= 2e-5 * big).all(), float((err / np.maximum(big, 1e-30)).max())


@pytest.mark.gpu
@pytest.mark.parametrize("where", ["k_nan", "k_inf", "q_nan", "v_inf", "v_nan"])
@pytest.mark.parametrize("rows,L,heads,kv,trim", [(5, 333, 8, 2, True), (9, 250, 4, 2, False),
                                                  (6, 481, 3, 3, False)])
def test_split_nonfinite_gpu(gpu_ctx, rows, L, heads, kv, trim, where):
    print(f"[split] {rows} x {L}, heads {heads}/{kv}, {where}", flush=True)
    hd = 256
    rng = Lcg(rows + L)
    q, gate = (rng.normal(rows * heads * hd * L).astype(np.float32).reshape(rows, -1, L) for _ in range(2))
    k, v = (rng.normal(rows * kv * hd * L).astype(np.float32).reshape(rows, -1, L) for _ in range(2))
    qn, kn = ((rng.normal(hd) * 0.1).astype(np.float32) for _ in range(2))
    mask = np.ones((rows, L), np.float32)
    for r in range(rows):
        mask[r, :17 * r] = 0.0
    mask[:, L // 2] = 0.0
    bad = np.nan if where.endswith("nan") else np.inf
    if where[0] == "q":
        q[1, 5, 140] = bad
    else:
        x = k if where[0] == "k" else v
        x[1, 7, 120] = bad              # kept from query 120 on
        x[2, 9, L // 2] = bad           # masked keys: must not leak
        x[3, hd + 3, 20] = -bad         # left padding
    args = tuple(t.reshape(-1) for t in (q, k, v, gate, qn, kn, mask)) + (rows, L, heads, kv, hd, 64,
                                                                         1.0e7, 1.0e-6)
    oracle.set_threads(8)
    with np.errstate(all="ignore"):
        want = oracle.jeff_rows(*args, trim_leading=trim)
    got = np.asarray(te.jeff_full_attention_rows(*args, trim_leading=trim, ctx=gpu_ctx))
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isposinf(got), np.isposinf(want))
    assert np.array_equal(np.isneginf(got), np.isneginf(want))
    ok = np.isfinite(want)  # a score that is not finite weighs 0
    assert ok.all() == (where[0] != "v")
    assert float(np.abs(got[ok] - want[ok]).max()) <= 2e-5
