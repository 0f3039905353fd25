"""Jeff rows (f32, head dims of the 256-wide kernels) where keys and values differ
by far more than a half-precision number's range: a masked key inside the sequence,
left padding, a key in the causal future, a key of almost no probability before all
others, one feature of V, and one feature of K that every query's zero meets, each
1e6, 1e12 or 3e38 times the rest; and norm weights that make scores past 2^24. Grids
above two workgroups per CU with 4, 2 and 1 query heads per workgroup, one of each
kernel for smaller grids, and a small head dim.

The expectation is the same formula in 64 bits (RoPE factors from the oracle's f32
table). An f32 evaluation is off by a few 2^-24 of sum_k p_k |v_k| of the
same output feature, plus as much for scores of order 33 (2^-24 x 33 x log2 e
each): the tolerance is the ops' 2e-5 of that sum, for each output by itself.
"""
import numpy as np
import pytest

import oracle
import tenferro_ext as te
from tenferro_ext.workloads import Lcg

THETA, EPS = 1.0e7, 1.0e-6
SHAPES = [(5, 333, 8, 2, 256, 64), (9, 250, 4, 2, 256, 64), (6, 481, 3, 3, 256, 32),
          (7, 289, 6, 2, 200, 50), (1, 200, 8, 2, 256, 64), (2, 200, 8, 2, 256, 64),
          (3, 120, 4, 2, 64, 32)]


def reference(q, k, v, gate, qn, kn, mask, rot, trim):
    """q, gate (R, H, hd, L), k, v (R, KV, hd, L): the output and sum_k p |v|, gated."""
    R, H, hd, L = q.shape
    KV = k.shape[1]
    out, size = np.zeros((2, R, H, hd, L))
    cos, sin = (t.reshape(L, rot // 2).astype(np.float64) for t in oracle.rope_table(L, rot, THETA))

    def prepared(x, w):
        x = x.T.astype(np.float64)
        with np.errstate(all="ignore"):
            x = x / np.sqrt((x * x).mean(1, keepdims=True) + np.float64(np.float32(EPS))) * (1.0 + w)
        n, h = len(x), rot // 2
        a, b, rest = x[:, :h], x[:, h:rot], x[:, rot:]
        return np.concatenate((a * cos[:n] - b * sin[:n], a * sin[:n] + b * cos[:n], rest), 1)

    for r in range(R):
        active = mask[r] != 0
        t0 = int(np.argmax(active)) if trim and active.any() else 0
        t = np.arange(t0, L)
        allowed = (t[None, :] <= t[:, None]) & active[None, t0:]
        for h in range(H):
            g = h * KV // H
            s = prepared(q[r, h, :, t0:], qn) @ prepared(k[r, g, :, t0:], kn).T / np.sqrt(hd)
            s = np.where(allowed, s, -np.inf)
            p = np.exp(s - np.where(allowed.any(1), s.max(1), 0.0)[:, None])
            p /= np.maximum(p.sum(1, keepdims=True), 1e-300)
            x = v[r, g, :, t0:].T.astype(np.float64)
            sg = 1.0 / (1.0 + np.exp(-gate[r, h, :, t0:].T.astype(np.float64)))
            out[r, h, :, t0:] = (p @ x * sg).T
            size[r, h, :, t0:] = (p @ np.abs(x) * sg).T
    return out, size


def inputs(R, L, H, KV, hd, case, big):
    rng = Lcg(R * 1000 + L + len(case))

    def normal(*shape):
        return rng.normal(int(np.prod(shape))).astype(np.float32).reshape(shape)

    q, gate, k, v = normal(R, H, hd, L), normal(R, H, hd, L), normal(R, KV, hd, L), normal(R, KV, hd, L)
    qn, kn = normal(hd) * np.float32(0.1), normal(hd) * np.float32(0.1)
    mask = np.ones((R, L), np.float32)
    for r in range(R):
        mask[r, :(37 * r) % max(L // 2, 1)] = 0.0
    large = np.float32(big) * (normal(2, R, KV, hd) % np.float32(1.0))
    if case == "masked":
        at = 3 * L // 4
        mask[:, at] = 0.0
        k[..., at], v[..., at] = large
    elif case == "padding":
        for r in range(R):
            n = (37 * r) % (L // 2)
            k[r, :, :, :n], v[r, :, :, :n] = large[0, r, :, :, None], large[1, r, :, :, None]
    elif case == "future":
        v[..., 3 * L // 4] = large[1]
    elif case == "improbable":  # the row's first key: its score is 33 below the others'
        qn[:], kn[:] = 0.5, 0.5
        q[:, :, hd // 2] = 40.0
        for r in range(R):
            at = (37 * r) % (L // 2)
            k[r, :, hd // 2, at] = -1e4
            v[r, :, :, at] = large[1, r] * np.float32(2.0 ** -20)
    elif case == "scores":      # far past 2^24: every query keeps its largest alone
        qn[:], kn[:] = big, big
    elif case == "feature_v":
        v[:, :, 3] *= np.float32(big)
    else:                       # feature_k, outside the rotated ones
        q[:, :, hd // 2] = 0.0
        k[:, :, hd // 2] *= np.float32(min(big, 1e6))
    return q, k, v, gate, qn, kn, mask


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["masked", "padding", "future", "improbable", "scores", "feature_v", "feature_k"])
@pytest.mark.parametrize("rows,L,heads,kv,hd,rot", SHAPES)
def test_ranges_gpu(gpu_ctx, rows, L, heads, kv, hd, rot, case):
    for big in {"masked": (1e6, 1e12, 3e38), "padding": (1e6, 1e12, 3e38), "scores": (3e3, 1e5, 1e9)}.get(
            case, (1e6, 1e12)):
        for trim in (False, True) if case == "padding" else (False,):
            print(f"[ranges] Jeff {rows} x {L}, heads {heads}/{kv} x {hd} {case} {big:g} {trim}", flush=True)
            x = inputs(rows, L, heads, kv, hd, case, big)
            want, size = reference(*x, rot, trim)
            q, k, v, gate, qn, kn, mask = (np.ascontiguousarray(t).reshape(-1) for t in x)
            got = te.jeff_full_attention_rows(q, k, v, gate, qn, kn, mask, rows, L, heads, kv, hd, rot,
                                              THETA, EPS, trim_leading=trim, ctx=gpu_ctx)
            err = np.abs(np.asarray(got).reshape(want.shape) - want)
            assert np.isfinite(err).all()
            ratio = float((err / np.maximum(size, 1e-300)).max())
            assert (err <= 2e-5 * size).all(), ratio


@pytest.mark.gpu
def test_bf16_scores_gpu(gpu_ctx):
    """Rows that keep their last key alone, under norm weights of 1e5: that key's value
    times the gate for the last query, 0 for the others."""
    print("[ranges] Jeff bf16 scores", flush=True)
    rows, L, heads, kv, hd = 16, 8, 8, 2, 256
    q, k, v, gate, qn, kn, mask = inputs(rows, L, heads, kv, hd, "scores", 1e5)
    mask[:, :L - 1], mask[:, L - 1] = 0.0, 1.0
    bits = [te.to_bf16_bits(t.reshape(-1)) for t in (q, k, v, gate)]
    v, gate = (te.bf16_bits_to_f32(b).astype(np.float64) for b in bits[2:])
    want = np.repeat(v.reshape(rows, kv, hd, L), heads // kv, axis=1) / (1.0 + np.exp(-gate.reshape(rows, heads, hd, L)))
    want[..., :L - 1] = 0.0
    got = np.asarray(te.jeff_full_attention_rows(*bits, qn, kn, mask.reshape(-1), rows, L, heads, kv, hd, 64,
                                                 THETA, EPS, bf16=True, ctx=gpu_ctx)).reshape(want.shape)
    assert np.isfinite(got).all() and float(np.abs(got - want).max()) <= 1e-2
