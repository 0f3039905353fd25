"""The model's linears over few columns (skinny_gemm.hip) at the sizes where
its tiles can go wrong: one to 160 packed columns (64 at hidden sizes above 768) (one or two column blocks,
partly filled), feature counts that are no multiple of 16 or 32, columns
longer than one batch of loads (LayerNorm in registers up to 768 and up to
1024), GeGLU halves that end inside a row block, norm biases, and weights at
an address that is only 4-byte aligned (the f32 GEMM takes those). Against the
oracle, with test_laya_model's tolerances (4 f32 layers: 1e-4 at d >= 256).
"""
import numpy as np
import pytest

from oracle import laya_model as om
from tenferro_ext.laya_model import LayaModel
from tenferro_ext.workloads import laya_model_batch, laya_model_checkpoint


def check(model, ck, batch, tol):
    want = om.forward(ck.encoder, ck.agent.action_count(), ck.weights, ck.head_heads, *batch)
    for got, ref in zip(model.forward(*batch), want):
        assert np.isfinite(got).all()
        err = float(np.abs(got - ref).max())
        assert err <= tol, f"max abs error {err} > {tol}"


@pytest.mark.gpu
@pytest.mark.parametrize("d,heads,inter,layers,L,B", [
    (36, 2, 20, 3, 7, 1), (96, 4, 100, 2, 17, 1), (768, 12, 1152, 2, 96, 1), (780, 6, 1156, 2, 30, 2),
    (1024, 16, 1300, 1, 16, 4), (264, 4, 400, 2, 80, 2), (264, 4, 400, 2, 81, 2)])
def test_small_forward_gpu(gpu_ctx, d, heads, inter, layers, L, B):
    print(f"[skinny] d {d} inter {inter} L {L} B {B}", flush=True)
    ck = laya_model_checkpoint(hidden=d, intermediate=inter, layers=layers, heads=heads, seed=d + L)
    batch = laya_model_batch(L, B, 3, 263, min_len=max(4, L - 5))
    check(LayaModel(ck, ctx=gpu_ctx), ck, batch, 2e-5 if d < 256 else 1e-4)


@pytest.mark.gpu
def test_unaligned_weights_gpu(gpu_ctx):
    """One weight shifted by four bytes: the forward takes the general linears."""
    import torch

    print("[skinny] unaligned weight", flush=True)
    ck = laya_model_checkpoint(hidden=64, intermediate=96, layers=2, heads=2, seed=5)
    model = LayaModel(ck, ctx=gpu_ctx)
    w = ck.weights["layers.1.wqkv.w"]
    room = torch.empty(w.size + 1, dtype=torch.float32, device="cuda")
    room[1:] = torch.from_numpy(w).cuda()
    torch.cuda.synchronize()
    model._layers[1].wqkv = room[1:].data_ptr()
    check(model, ck, laya_model_batch(20, 2, 3, 263, min_len=12), 2e-5)
