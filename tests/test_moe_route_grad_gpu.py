"""Gradients of a routed layer's glue."""
import pytest
import torch

from areal_vllm_amd import ops

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,k,H", [(1, 1, 8), (3, 2, 2040), (5, 3, 2048), (2, 4, 2056), (64, 8, 2048), (7, 9, 4104), (3, 16, 64)])
def test_recombination_backward_is_that_of_the_two_passes(T, k, H):
    """Rows bit for bit; a weight's gradient against 64 bits: H products summed in fp32, rounded once."""
    g = torch.Generator(device=DEV).manual_seed(H + k)
    inv = torch.randperm(T * k, device=DEV, generator=g)
    order = torch.argsort(inv)
    ys = torch.randn(T * k, H, device=DEV, generator=g).bfloat16().requires_grad_(True)
    w = torch.rand(T, k, device=DEV, generator=g).requires_grad_(True)
    do = torch.randn(T, H, device=DEV, generator=g).bfloat16()
    dys, dw = torch.autograd.grad(ops.moe_combine(ys, w, order, inv), (ys, w), do)
    (only,) = torch.autograd.grad(ops.moe_combine(ys, w.detach(), order, inv), (ys,), do)
    assert torch.equal(dys, only)
    want = (ys.detach().double()[inv].view(T, k, H) * do.double().unsqueeze(1)).sum(-1)
    size = (ys.detach().double()[inv].view(T, k, H) * do.double().unsqueeze(1)).abs().sum(-1)
    assert bool(((dw.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -20 * size).all())
