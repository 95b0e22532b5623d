"""LM head + log-prob: the backward over all rows at once against float64, beside the backward chunk by chunk."""
import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.ops import train_gemm as tg

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


# one launch for all rows (V a multiple of 128; from 8192 on both gradients are the own kernels', split over V); chunk by chunk where
# they do not take the shape; padded rows
@pytest.mark.parametrize("T,V,chunk", [(1300, 8320, 512), (600, 9088, 256), (1300, 2176, 512), (1024, 2176, 512), (700, 2056, 256), (700, 2055, 256), (300, 2176, 512)])
def test_backward_of_several_chunks(T, V, chunk):
    H = 256
    assert tg._dgrad_own(T, V, H) == (V >= 8192)
    g = torch.Generator(device=DEV).manual_seed(T + V)
    h = torch.randn(T, H, device=DEV, generator=g).bfloat16()
    w = (torch.randn(V, H, device=DEV, generator=g) / H ** 0.5).bfloat16()
    labels = torch.randint(0, V, (T,), device=DEV, generator=g)
    a, b = torch.randn(T, device=DEV, generator=g) / T, torch.randn(T, device=DEV, generator=g) / T

    h64, w64 = h.double().requires_grad_(True), w.double().requires_grad_(True)
    lp = torch.log_softmax(h64 @ w64.t(), -1)
    ((lp.gather(1, labels[:, None])[:, 0] * a).sum() + (-(lp.exp() * lp).sum(-1) * b).sum()).backward()

    hx, wx = h.clone().requires_grad_(True), w.clone().requires_grad_(True)
    wx.main_grad = torch.ones(V, H, device=DEV)  # what earlier micro-batches have left
    logp, ent = ops.lm_head_logprobs(hx, wx, labels, chunk=chunk)
    ((logp * a).sum() + (ent * b).sum()).backward()
    # logits and their gradients are held in bf16: 2^-9 relative each
    for got, want in ((hx.grad, h64.grad), (wx.main_grad - 1.0, w64.grad)):
        assert float((got.double() - want).norm() / want.norm()) < 2.0 ** -7
