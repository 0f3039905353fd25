"""Laya attention where keys and values differ by far more than a half-precision
number's range inside one 32-key tile: a masked key, a key that one query of a
workgroup keeps, a key outside the other queries' window, one feature of V, one
feature of K that every query's zero meets, and a key of almost no probability,
each 1e6, 1e12 or 3e38 times the rest; and scores of that size. For every workgroup shape (two and four
waves per team, one team) and head dim of the aligned path, both entries.

The expectation is the same formula in 64 bits (RoPE factors from the oracle's f32
table). An f32 evaluation is off by a few 2^-24 of sum_k p_k |v_k| of the
same output feature, plus as much for scores of order 30 (2^-24 x 30 x log2 e
each): the tolerance is the ops' 2e-5 of that sum, for each output by itself.
"""
import numpy as np
import pytest

import oracle
import tenferro_ext as te
from tenferro_ext.workloads import Lcg

BASE = 160000.0
SHAPES = [(64, 2, 90, 1), (64, 2, 333, 2), (64, 12, 200, 4), (64, 12, 333, 4), (32, 3, 200, 2),
          (128, 4, 290, 2), (128, 12, 333, 4)]


def reference(qkv, keep, heads, rope):
    """qkv (B, L, 3d), keep (B, key, query): the output and sum_k p |v|, (B, L, d)."""
    B, L, d3 = qkv.shape
    d = d3 // 3
    hd = d // heads
    x = qkv.astype(np.float64)
    out, size = np.zeros((2, B, L, d))
    cos, sin = (t.reshape(L, hd // 2).astype(np.float64) for t in oracle.rope_table(L, hd, BASE))

    def rotate(t):
        a, b = t[:, :hd // 2], t[:, hd // 2:]
        return np.concatenate((a * cos - b * sin, a * sin + b * cos), 1) if rope else t

    for b in range(B):
        for h in range(heads):
            q, k, v = (x[b, :, j * d + h * hd:j * d + (h + 1) * hd] for j in range(3))
            with np.errstate(all="ignore"):
                s = rotate(q) @ rotate(k).T / np.sqrt(hd)
            s = np.where(keep[b].T != 0, s, -np.inf)
            p = np.exp(s - s.max(1, keepdims=True))
            p /= p.sum(1, keepdims=True)
            out[b, :, h * hd:(h + 1) * hd] = p @ v
            size[b, :, h * hd:(h + 1) * hd] = p @ np.abs(v)
    return out, size


def inputs(hd, heads, L, B, case, big):
    """(qkv, valid, window, keep): keep None where valid and window say it all."""
    rng = Lcg(hd + L + len(case))
    d = hd * heads
    x = rng.normal(3 * d * L * B).astype(np.float32).reshape(B, L, 3, heads, hd)
    valid, window, keep = np.ones((B, L), np.uint8), -1, None
    large = np.float32(big) * (rng.normal(2 * d).reshape(2, heads, hd) % 1.0).astype(np.float32)
    if case == "masked":      # in a tile that is kept otherwise
        valid[:, 37] = 0
        x[:, 37, 1:] = large
    elif case == "window":    # kept by the 41 queries around it
        window = 20
        x[:, 37, 2] = large[1]
    elif case == "one_query":
        keep = np.ones((B, L, L), np.uint8)
        keep[:, 70, :] = 0
        keep[:, 70, 75] = 1
        x[:, 70, 2] = large[1]
    elif case == "scores":    # far past 2^24, one or two keys each
        keep = np.zeros((B, L, L), np.uint8)
        t = np.arange(L)
        keep[:, t, t] = 1
        keep[:, (t + 7) % L, t] = t % 3 > 0
        x[:, :, :2] *= np.float32(big) ** np.float32(0.5)
    elif case == "feature_v":
        x[:, :, 2, :, 3] *= np.float32(big)
    elif case == "feature_k":  # a RoPE pair
        pair = [5, 5 + hd // 2]
        x[:, :, 0, :, pair] = 0.0
        x[:, :, 1, :, pair] *= np.float32(big)
    else:                      # improbable: a pair that hardly turns takes key 2's score down by 50 or more
        slow = hd // 2 - 1
        x[:, :, 0, :, slow] = 20.0
        x[:, 2, 1, :, slow] = -50.0 * np.sqrt(hd) / 20.0 - 12.0
        x[:, 2, 2] = large[1]
    return x.reshape(B, L, 3 * d), valid, window, keep


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["masked", "window", "one_query", "scores", "feature_v", "feature_k", "improbable"])
@pytest.mark.parametrize("hd,heads,L,B", SHAPES)
def test_ranges_gpu(gpu_ctx, hd, heads, L, B, case):
    d = hd * heads
    for big in {"masked": (1e6, 1e12, 3e38), "window": (1e6, 1e12, 3e38), "scores": (1e9, 1e12, 1e18)}.get(
            case, (1e6, 1e12)):
        print(f"[ranges] Laya hd {hd} heads {heads} L {L} B {B} {case} {big:g}", flush=True)
        qkv, valid, window, keep = inputs(hd, heads, L, B, case, big)
        flat = np.ascontiguousarray(qkv.reshape(-1))
        bits = keep if keep is not None else oracle.laya_build_mask(valid.reshape(-1), L, B, window)
        want, size = reference(qkv, bits.reshape(B, L, L), heads, True)
        got = [te.laya_attention_block(flat, bits.reshape(-1), d, heads, BASE,
                                       qkv_shape=(3 * d, L, B), ctx=gpu_ctx)]
        if keep is None:
            got.append(te.laya_attention_structured(flat, valid.reshape(-1), d, heads, L, B, window,
                                                    BASE, ctx=gpu_ctx))
            # Their key spans differ; a query's bits follow from the keys it keeps alone.
            assert np.array_equal(np.asarray(got[0]), np.asarray(got[1]))
        for g in got:
            err = np.abs(np.asarray(g).reshape(B, L, d) - want)
            assert np.isfinite(err).all()
            assert (err <= 2e-5 * size).all(), float((err / size).max())
