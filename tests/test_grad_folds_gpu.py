"""Gradients of biases and norm weights that their kernels add to the fp32 buffer behind the parameter."""
import pytest
import torch

from areal_vllm_amd import ops

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


def _parameter(t):
    p = torch.nn.Parameter(t.bfloat16())
    p.main_grad = torch.full(t.shape, 3.0, device=DEV)
    p.told = 0

    def told(q):
        q.told += 1

    p._after_fold = told
    return p


@pytest.mark.parametrize("M", [1, 31, 32, 33, 256, 257, 1024, 1025, 1536, 40000])
@pytest.mark.parametrize("N", [8, 64, 72, 2048])
@pytest.mark.parametrize("strided", [False, True])
def test_bias(M, N, strided):
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x = torch.randn(M, 64, device=DEV, generator=g).bfloat16().requires_grad_(True)
    w, b = _parameter(torch.randn(N, 64, device=DEV, generator=g)), _parameter(torch.randn(N, device=DEV, generator=g))
    dy = torch.randn(M, N + (8 if strided else 0), device=DEV, generator=g).bfloat16()[:, :N]
    ops.linear(x, w, b).backward(dy)
    assert b.grad is None and b.told == 1 and w.told == 1
    want = dy.double().sum(0) + 3.0
    # fp32 sums of M values: the buffer's own rounding and sqrt(M) of those of the sums' size
    assert float((b.main_grad.double() - want).abs().max()) < 2.0 ** -22 * (3.0 + M ** 0.5 * 8)


def test_bias_that_the_kernel_does_not_take():
    x = torch.randn(40, 64, device=DEV).bfloat16().requires_grad_(True)
    w, b = _parameter(torch.randn(12, 64, device=DEV)), _parameter(torch.randn(12, device=DEV))  # no multiple of 8 columns
    dy = torch.randn(40, 12, device=DEV).bfloat16()
    ops.linear(x, w, b).backward(dy)
    assert b.told == 0 and torch.allclose(b.grad.float(), dy.float().sum(0), rtol=2.0 ** -7, atol=0.05)
    b2 = torch.nn.Parameter(torch.randn(16, device=DEV).bfloat16())  # no buffer behind it
    w2 = _parameter(torch.randn(16, 64, device=DEV))
    ops.linear(x, w2, b2).backward(torch.ones(40, 16, device=DEV).bfloat16())
    assert torch.equal(b2.grad.float(), torch.full((16,), 40.0, device=DEV))


@pytest.mark.parametrize("T,H", [(1, 8), (5, 1536), (700, 1536), (4097, 256), (3000, 8192)])
@pytest.mark.parametrize("residual,gemma", [(False, False), (True, True)])
def test_norm_weight(T, H, residual, gemma):
    g = torch.Generator(device=DEV).manual_seed(T + H)
    x = torch.randn(T, H, device=DEV, generator=g).bfloat16().requires_grad_(True)
    r = torch.randn(T, H, device=DEV, generator=g).bfloat16().requires_grad_(True) if residual else None
    w = _parameter(torch.rand(H, device=DEV, generator=g) + 0.5)
    plain = torch.nn.Parameter(w.detach().clone())
    dy = torch.randn(T, H, device=DEV, generator=g).bfloat16()
    dx = []
    for p in (w, plain):
        x.grad = None
        ops.rmsnorm(x, p, 1e-6, r, gemma)[0].backward(dy)
        dx.append(x.grad.clone())
    assert torch.equal(*dx) and w.grad is None and w.told == 1
    got = w.main_grad.double() - 3.0  # the sum that is rounded to 16 bits where it goes back through autograd
    assert float((got - plain.grad.double()).abs().max()) <= float((2.0 ** -8 * got.abs() + 2.0 ** -20).max())
    s = x.detach().double() if r is None else (x.detach().float() + r.detach().float()).bfloat16().double()
    want = (dy.double() * s * torch.rsqrt(s.pow(2).mean(-1, keepdim=True) + 1e-6)).sum(0)
    assert float((got - want).abs().max()) < 2.0 ** -20 * (4.0 + T ** 0.5 * 8)
