"""The layer and model linears on bf16 planes (split_gemm.hip), at the sizes
where the planes and tiles can go wrong: k and feature counts that are no
multiple of 32 or 16, columns that end inside a tile, odd question rows,
GeGLU halves that end inside a row block, rows that hold inf or NaN, and
operands whose scales only meet in the product.

Every shape here is large enough for that path (dims of 512, 384 columns, 9 * 2^27
products of a layer's square linear, 6 * 2^27 in the forward); the oracle's f32 layers
are the expectation. The planes hold every operand whole and their sums are f32,
so the layers' tolerance of 2e-5 on outputs of order 1 stays as it is.
"""
import numpy as np
import pytest

import oracle
import tenferro_ext as te
from tenferro_ext.workloads import (Lcg, jeff_layer_config, laya_model_batch,
                                    laya_model_checkpoint)

TOL = 2e-5


def same(got, want, tol=TOL):
    got, want = (np.asarray(a, np.float32).reshape(-1) for a in (got, want))
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf]) and np.array_equal(np.isinf(got), inf)
    ok = np.isfinite(want)
    err = float(np.abs(got[ok] - want[ok]).max())
    assert err <= tol, f"max abs error {err} > {tol}"


def laya_layer(d, heads, L, B, *, window=40):
    rng = Lcg(900 + d)
    valid = np.zeros((B, L), np.uint8)
    for b in range(B):
        valid[b, :L - 37 * b] = 1
    return dict(x=rng.normal(d * L * B).astype(np.float32),
                keep=oracle.laya_build_mask(valid.reshape(-1), L, B, window),
                w_in=(rng.normal(3 * d * d) * d ** -0.5).astype(np.float32),
                b_in=(rng.normal(3 * d) * 0.1).astype(np.float32),
                w_out=(rng.normal(d * d) * d ** -0.5).astype(np.float32),
                b_out=(rng.normal(d) * 0.1).astype(np.float32), hidden=d, heads=heads, length=L,
                batch=B, rope_base=10000.0)


def run_laya(ctx, c):
    return te.laya_attention_layer(c["x"], c["keep"], c["w_in"], c["b_in"], c["w_out"], c["b_out"],
                                   c["hidden"], c["heads"], c["length"], c["batch"],
                                   c["rope_base"], ctx=ctx)


@pytest.mark.gpu
@pytest.mark.parametrize("d,heads,L,B", [(520, 5, 951, 5), (544, 8, 1030, 4), (768, 12, 421, 5),
                                         (1056, 8, 109, 10)])
def test_laya_layer_tile_edges_gpu(gpu_ctx, d, heads, L, B):
    print(f"[split] Laya layer d {d} L {L} B {B}", flush=True)
    c = laya_layer(d, heads, L, B)
    same(run_laya(gpu_ctx, c), oracle.laya_attention_layer(**c))


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["x", "w_out", "scales"])
def test_laya_layer_values_gpu(gpu_ctx, case):
    """x: a token with an inf and one with a NaN (never kept as keys), so their
    columns alone are not finite. w_out: one inf weight makes its output
    feature +-inf by the sign of the attended feature. scales: V's weights
    times 2^60 and W_out's times 2^-60."""
    print(f"[split] Laya layer values: {case}", flush=True)
    d, L, B = 520, 951, 5
    c = laya_layer(d, 5, L, B)
    if case == "x":
        keep = c["keep"].reshape(B, L, L)
        x = c["x"].reshape(B, L, d)
        for b, t, value in ((0, 3, np.inf), (2, 100, np.nan), (1, 512, -np.inf)):
            x[b, t, 11] = value
            keep[b, t, :] = 0
    elif case == "w_out":
        c["w_out"][7 * d + 19] = np.inf
    else:
        c["w_in"][2 * d * d:] *= np.float32(2.0 ** 60)
        c["b_in"][2 * d:] *= np.float32(2.0 ** 60)
        c["w_out"] *= np.float32(2.0 ** -60)
    with np.errstate(all="ignore"):
        want = oracle.laya_attention_layer(**c)
    same(run_laya(gpu_ctx, c), want)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,length,hidden", [(4, 291, 520), (3, 420, 528)])
def test_jeff_layer_tile_edges_gpu(gpu_ctx, rows, length, hidden):
    print(f"[split] Jeff layer {rows} x {length}, hidden {hidden}", flush=True)
    oracle.set_threads(8)
    j = jeff_layer_config(4, rows=rows, length=length, hidden=hidden)
    args = (j.x, j.w_q, j.w_gate, j.w_k, j.w_v, j.w_o, j.q_norm, j.k_norm, j.mask)
    dims = (j.rows, j.length, j.hidden, j.heads, j.kv_heads, j.head_dim, j.rotary_dim, j.theta,
            j.eps)
    want = oracle.jeff_layer_rows(*args, *dims, trim_leading=True)
    same(te.jeff_full_attention_layer_rows(*args, *dims, trim_leading=True, ctx=gpu_ctx), want)


@pytest.mark.gpu
@pytest.mark.parametrize("d,inter", [(512, 516), (520, 600)])
def test_forward_tile_edges_gpu(gpu_ctx, d, inter):
    """GeGLU halves that end inside a 16-row block, packed columns of padded prompts."""
    from oracle import laya_model as om
    from tenferro_ext.laya_model import LayaModel

    print(f"[split] forward d {d} inter {inter}", flush=True)
    ck = laya_model_checkpoint(hidden=d, intermediate=inter, layers=2, heads=8 if d == 512 else 5, seed=d)
    batch = laya_model_batch(431, 9, 4, 263, min_len=400)
    oracle.set_threads(8)
    logits, action = LayaModel(ck, ctx=gpu_ctx).forward(*batch)
    want = om.forward(ck.encoder, ck.agent.action_count(), ck.weights, ck.head_heads, *batch)
    for got, ref in zip((logits, action), want):
        same(got, ref, 1e-4)  # as test_laya_model's wide random model: 2 encoder layers' roundings
