"""The layer and model linears where elements of one row differ by far more than a
half-precision number's range: a feature of the tokens that meets zero weights, a
weight column that meets zero features, a large feature met by correspondingly
small weights, and the same in the output projection and behind a LayerNorm.

Laya: every token keeps only itself, so the attention returns V; Jeff: rows of one
token, V times the gate's sigmoid. The expectation is the product in 64 bits. An f32
sum of k <= 544 terms in any order stays within k 2^-24 of sum |w||x|, in
practice within sqrt(k) 2^-24 x 1.5 = 2e-6 of it; two linears in a row: 4e-6 of the sum
over both. The forward: the oracle's f32 model, with test_split_linears' tolerance.
"""
import numpy as np
import pytest

import oracle
import tenferro_ext as te
from tenferro_ext.workloads import Lcg, laya_model_batch, laya_model_checkpoint

TOL = 4e-6


def spread(case, big, x, w_in, w_out, at):
    """Widens one feature of x (n, k), w_in (v, k) or w_out (out, v) in place."""
    big = np.float32(big)
    if case == "token":          # meets zero weights
        x[:, at] *= big
        w_in[:, at] = 0.0
    elif case == "weight":       # meets zero features
        w_in[:, at] *= big
        x[:, at] = 0.0
    elif case == "both":         # meets small weights
        x[:, at] *= big
        w_in[:, at] /= big
    else:                        # w_out: meets attended zeros
        w_out[:, at] *= big
        w_in[at] = 0.0


CASES = [(c, b) for c in ("token", "weight", "both", "w_out") for b in (2.0 ** 24, 1e12)]


@pytest.mark.gpu
@pytest.mark.parametrize("case,big", CASES)
@pytest.mark.parametrize("d,heads,L,B", [(512, 8, 640, 8), (520, 5, 613, 8)])
def test_laya_layer_ranges_gpu(gpu_ctx, d, heads, L, B, case, big):
    print(f"[ranges] Laya layer d {d} L {L} B {B} {case} {big:g}", flush=True)
    rng = Lcg(d + L)
    x = rng.normal(B * L * d).astype(np.float32).reshape(B * L, d)
    w_in = (rng.normal(3 * d * d) * d ** -0.5).astype(np.float32).reshape(3 * d, d)
    w_out = (rng.normal(d * d) * d ** -0.5).astype(np.float32).reshape(d, d)
    w_v = w_in[2 * d:]
    spread(case, big, x, w_v, w_out, 7)
    if case in ("token", "both"):
        w_in[:2 * d, 7] = 0.0
    keep = np.broadcast_to(np.eye(L, dtype=np.uint8), (B, L, L))
    got = te.laya_attention_layer(x.reshape(-1), np.ascontiguousarray(keep).reshape(-1),
                                  w_in.reshape(-1), None, w_out.reshape(-1), None, d, heads, L, B,
                                  10000.0, ctx=gpu_ctx)
    x, w_v, w_out = (t.astype(np.float64) for t in (x, w_v, w_out))
    want = x @ w_v.T @ w_out.T
    size = np.abs(x) @ np.abs(w_v).T @ np.abs(w_out).T
    err = np.abs(np.asarray(got).reshape(B * L, d) - want)
    assert (err <= TOL * size).all(), float((err / size).max())


@pytest.mark.gpu
@pytest.mark.parametrize("case,big", CASES)
def test_jeff_layer_ranges_gpu(gpu_ctx, case, big):
    print(f"[ranges] Jeff layer {case} {big:g}", flush=True)
    R, n, heads, kv, hd = 4410, 544, 8, 4, 64
    W, KW = heads * hd, kv * hd
    rng = Lcg(n)
    x = rng.normal(R * n).astype(np.float32).reshape(R, n)
    w_q, w_gate, w_k, w_v = ((rng.normal(o * n) * n ** -0.5).astype(np.float32).reshape(o, n)
                             for o in (W, W, KW, KW))
    w_o = (rng.normal(n * W) * W ** -0.5).astype(np.float32).reshape(n, W)
    spread(case, big, x, w_v, w_o[:, :hd], 7)
    if case == "w_out":  # the other query head of kv head 0
        w_o[:, hd + 7] = w_o[:, 7]
    if case in ("token", "both"):
        for w in (w_q, w_gate, w_k):
            w[:, 7] = 0.0
    one = np.ones(R, np.float32)
    norm = np.zeros(hd, np.float32)
    got = te.jeff_full_attention_layer_rows(
        x.reshape(-1), w_q.reshape(-1), w_gate.reshape(-1), w_k.reshape(-1), w_v.reshape(-1),
        w_o.reshape(-1), norm, norm, one, R, 1, n, heads, kv, hd, 32, 1.0e7, 1.0e-6, ctx=gpu_ctx)
    x, w_gate, w_v, w_o = (t.astype(np.float64) for t in (x, w_gate, w_v, w_o))
    sig = 1.0 / (1.0 + np.exp(-(x @ w_gate.T)))

    def expand(v):
        return np.repeat(v.reshape(R, kv, 1, hd), heads // kv, axis=2).reshape(R, W)

    v, v_size = expand(x @ w_v.T), expand(np.abs(x) @ np.abs(w_v).T)
    want = (v * sig) @ w_o.T
    # sigmoid' <= sigmoid: the gate's own sum counts once more
    size = (v_size * sig * (1.0 + np.abs(x) @ np.abs(w_gate).T)) @ np.abs(w_o).T
    err = np.abs(np.asarray(got).reshape(R, n) - want)
    assert (err <= TOL * size).all(), float((err / np.maximum(size, 1e-300)).max())


@pytest.mark.gpu
@pytest.mark.parametrize("big", [2.0 ** 24, 1e12])
def test_forward_ranges_gpu(gpu_ctx, big):
    """One feature of every LayerNorm's output big, where all weights after it are 0."""
    from oracle import laya_model as om
    from tenferro_ext.laya_model import LayaModel

    print(f"[ranges] forward {big:g}", flush=True)
    d = 512
    ck = laya_model_checkpoint(hidden=d, intermediate=516, layers=2, heads=8, seed=3)
    w = ck.weights
    for norm, linear in (("layers.1.attn_norm", "layers.1.wqkv"), ("layers.0.mlp_norm", "layers.0.wi"),
                         ("layers.1.mlp_norm", "layers.1.wi"), ("head.0.norm1", "head.0.in_proj"),
                         ("head.0.norm2", "head.0.linear1")):
        w[norm + ".w"][9] = big
        w[linear + ".w"].reshape(-1, d)[:, 9] = 0.0
    batch = laya_model_batch(431, 9, 4, 263, min_len=400)
    oracle.set_threads(8)
    want = om.forward(ck.encoder, ck.agent.action_count(), w, ck.head_heads, *batch)
    for got, ref in zip(LayaModel(ck, ctx=gpu_ctx).forward(*batch), want):
        assert np.isfinite(got).all()
        assert float(np.abs(got - ref).max()) <= 1e-4
