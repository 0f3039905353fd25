"""Laya attention with keys and values whose magnitude changes from tile to
tile: jumps up and down by far more than a half-precision number holds, all-zero
tiles, a tile with an inf that is never kept, in both entries, for every
workgroup shape (teams of two and four waves, one team) and head dim of the
aligned path (test_laya_ranges has the jumps inside a tile). The expectation is
the oracle, which takes its RoPE angles in f32 as the op does (64-bit brute force
does not: at position 417 an angle differs by up to 417 * 2^-24, and scores of
order 30 by as much times that, far above the tolerance). An output is a convex combination of kept
values, so the tolerance is 2e-5 of the largest value a query keeps (its
window), the f32 tolerance at that scale.
"""
import numpy as np
import pytest

import oracle
import tenferro_ext as te
from tenferro_ext.workloads import Lcg

WINDOW = 20


def case(hd, heads, L, B, seed):
    rng = Lcg(seed)
    d = hd * heads
    qkv = rng.normal(3 * d * L * B).astype(np.float32).reshape(B, L, 3 * d)
    # per 32-key tile: K * 2^a (q scaled back so that scores stay of order 1
    # where both meet), V * 2^b
    up = [0, -18, 12, 0, 30, -30, 3, 60, -60, 0, 9, -9]
    for t in range((L + 31) // 32):
        sl = slice(32 * t, 32 * t + 32)
        qkv[:, sl, d:2 * d] *= np.float32(2.0 ** min(up[(t + 2) % len(up)], 3))
        qkv[:, sl, 2 * d:] *= np.float32(2.0 ** up[t % len(up)])
    if L > 100:
        qkv[0, 64:96, d:] = 0.0  # a tile of zero keys and values
    valid = np.ones((B, L), np.uint8)
    if L > 40:
        valid[0, 37] = 0         # never kept
        qkv[0, 37, d + 3] = np.inf
        qkv[0, 37, 2 * d + 5] = np.inf
    return d, qkv, valid


@pytest.mark.gpu
@pytest.mark.parametrize("hd,heads,L,B", [(64, 2, 30, 1), (64, 2, 333, 2), (64, 12, 333, 4),
                                          (64, 12, 417, 8), (32, 3, 200, 2), (128, 4, 290, 4),
                                          (128, 12, 333, 8)])
def test_tile_scales_gpu(gpu_ctx, hd, heads, L, B):
    print(f"[scales] hd {hd} heads {heads} L {L} B {B}", flush=True)
    d, qkv, valid = case(hd, heads, L, B, 31 * hd + L)
    keep = oracle.laya_build_mask(valid.reshape(-1), L, B, WINDOW).reshape(B, L, L)
    keep[0, :, 37 if L > 40 else 0] = keep[0, :, 36 if L > 40 else 1]  # no query keeps a whole row
    flat = np.ascontiguousarray(qkv.reshape(-1))
    with np.errstate(all="ignore"):
        want = oracle.laya_attention_block(flat, keep.reshape(-1), d, heads, L, B, 10000.0)
    got = te.laya_attention_block(flat, keep.reshape(-1), d, heads, 10000.0,
                                  qkv_shape=(3 * d, L, B), ctx=gpu_ctx)
    got, want = np.asarray(got).reshape(B, L, d), want.reshape(B, L, d)
    assert np.isfinite(want).all() and np.isfinite(got).all()
    # the largest finite |v| each query keeps
    v = np.where(np.isfinite(qkv[..., 2 * d:]), np.abs(qkv[..., 2 * d:]), 0).max(-1)  # [b, key]
    big = np.stack([np.where(keep[b].astype(bool), v[b][:, None], 0).max(0) for b in range(B)])
    err = np.abs(got - want).max(-1)
    assert (err <= 2e-5 * big + 1e-30).all(), float((err / np.maximum(big, 1e-30)).max())
