"""RMSNorm backward around the row count from which the residual gradient is requested with the row, and every register class."""
import pytest
import torch

from areal_vllm_amd import ops

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 4096, 4097, 6001])
@pytest.mark.parametrize("H", [520, 1024, 1536, 2048, 2056, 4104])
@pytest.mark.parametrize("residual", [False, True])
def test_backward(T, H, residual):
    g = torch.Generator(device=DEV).manual_seed(T + H)
    x = torch.randn(T, H, device=DEV, generator=g).bfloat16().requires_grad_(True)
    r = torch.randn(T, H, device=DEV, generator=g).bfloat16().requires_grad_(True) if residual else None
    w = (1 + 0.1 * torch.randn(H, device=DEV, generator=g)).bfloat16().requires_grad_(True)
    dy, ds = (torch.randn(T, H, device=DEV, generator=g).bfloat16() for _ in range(2))
    y, s = ops.rmsnorm(x, w, 1e-6, r)
    torch.autograd.backward([y, s] if residual else [y], [dy, ds] if residual else [dy])
    sd, wd = s.detach().double(), w.detach().double()
    rstd = torch.rsqrt(sd.pow(2).mean(-1, keepdim=True) + 1e-6)
    xh, gd = sd * rstd, dy.double() * wd
    assert bool(((y.double() - xh * wd).abs() <= 2.0 ** -8 * (xh * wd).abs() + 1e-5).all())  # rounded to bf16 once
    dx = rstd * (gd - xh * (gd * xh).mean(-1, keepdim=True)) + (ds.double() if residual else 0.0)
    assert bool(((x.grad.double() - dx).abs() <= 2.0 ** -8 * dx.abs() + 1e-5).all())
    if residual:
        assert torch.equal(x.grad, r.grad)
    dw = (dy.double() * xh).sum(0)
    # one rounding to bf16, and fp32 sums of T products of size one
    assert bool(((w.grad.double() - dw).abs() <= 2.0 ** -8 * dw.abs() + 1e-6 * T ** 0.5 + 1e-5).all())
