"""Gradients of biases, norm weights and routers go through autograd, also where an fp32 buffer stands behind the parameter: what hangs on the
parameter sees them, and one backward pass reports each once."""
import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.models.config import ModelConfig
from areal_vllm_amd.models.transformer import MoE

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


def _parameter(t):
    p = torch.nn.Parameter(t.bfloat16())
    p.main_grad = torch.zeros(t.shape, device=DEV)
    p.told = 0

    def told(q):
        q.told += 1

    p._after_fold = told
    return p


def _bias():
    x = torch.ones(40, 64, device=DEV).bfloat16()
    w = torch.nn.Parameter(torch.zeros(16, 64, device=DEV).bfloat16())
    w.main_grad = torch.zeros(16, 64, device=DEV)
    b = _parameter(torch.zeros(16, device=DEV))
    return b, lambda: ops.linear(x, w, b), 40.0


def _norm():
    x = torch.ones(40, 64, device=DEV).bfloat16().requires_grad_(True)
    w = _parameter(torch.ones(64, device=DEV))
    return w, lambda: ops.rmsnorm(x, w, 0.0)[0], 40.0


@pytest.mark.parametrize("case", [_bias, _norm])
def test_hooks_and_direct_gradients(case):
    p, f, want = case()
    seen = []
    p.register_hook(lambda g: seen.append(g.clone()))
    y = f()
    y.backward(torch.ones_like(y))
    assert len(seen) == 1 and torch.equal(seen[0].float(), torch.full_like(p, want).float())
    assert torch.equal(p.grad, seen[0]) and not p.main_grad.any()
    (g,) = torch.autograd.grad(f(), p, torch.ones_like(y))
    assert torch.equal(g, seen[0])


@pytest.mark.parametrize("case", [_bias, _norm])
def test_a_parameter_used_twice_is_reported_once(case):
    p, f, want = case()
    calls = []
    p.register_post_accumulate_grad_hook(lambda q: calls.append(1))
    y = f() + f()
    y.backward(torch.ones_like(y))
    assert calls == [1] and p.told == 0 and torch.equal(p.grad.float(), torch.full_like(p, 2 * want).float())


@pytest.mark.parametrize("tokens", [5, 256, 1000])
def test_router(tokens):
    """The whole layer, of a size that the split weight-gradient product takes (from 256 tokens on)."""
    cfg = ModelConfig(family="qwen3_moe", vocab_size=64, hidden_size=256, n_layers=1, n_q_heads=2, n_kv_heads=1, head_dim=64,
                      intermediate_size=64, n_experts=128, n_experts_per_tok=2, moe_intermediate_size=64)
    layer = MoE(cfg, 1, torch.bfloat16, DEV)
    g = torch.Generator(device=DEV).manual_seed(tokens)
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, 0.05, generator=g)
    p = layer.router
    p.main_grad, p.told, seen, calls = torch.zeros(p.shape, device=DEV), 0, [], []
    p._after_fold = lambda q: setattr(q, "told", q.told + 1)
    p.register_hook(lambda t: seen.append(t.clone()))
    p.register_post_accumulate_grad_hook(lambda q: calls.append(1))
    x = torch.randn(tokens, 256, device=DEV, generator=g).bfloat16()
    dy = torch.randn(tokens, 256, device=DEV, generator=g).bfloat16()
    layer(x, None).backward(dy)
    assert calls == [1] and p.told == 0 and not p.main_grad.any() and torch.equal(p.grad, seen[0]) and bool(p.grad.any())
    (again,) = torch.autograd.grad(layer(x, None), p, dy)
    assert torch.equal(again, p.grad)


@pytest.mark.parametrize("T,E,H", [(255, 128, 256), (256, 128, 256), (1000, 256, 512), (4099, 128, 2048)])
@pytest.mark.parametrize("strided", [False, True])
def test_router_logits(T, E, H, strided):
    g = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn(T, H + 8 * strided, device=DEV, generator=g).bfloat16()[:, :H].requires_grad_(True)
    w = torch.nn.Parameter((torch.randn(E, H, device=DEV, generator=g) * 0.1).bfloat16())
    dy = torch.randn(T, E, device=DEV, generator=g).bfloat16()
    y = ops.router_logits(x, w)
    assert torch.equal(y, torch.nn.functional.linear(x, w))
    dx, dw = torch.autograd.grad(y, (x, w), dy)
    # fp32 sums of up to 4099 products of values of order one, rounded to 16 bits once
    for got, want in ((dw, dy.double().t() @ x.detach().double()), (dx, dy.double() @ w.detach().double())):
        assert float(((got.double() - want).abs() - 2.0 ** -8 * want.abs()).max()) < 2.0 ** -20 * T ** 0.5 * 8


@pytest.mark.parametrize("M", [1, 31, 32, 33, 256, 257, 1024, 1025, 1536, 40000])
@pytest.mark.parametrize("N", [8, 12, 64, 72, 2048])
@pytest.mark.parametrize("strided", [False, True])
def test_bias_values(M, N, strided):
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x = torch.randn(M, 64, device=DEV, generator=g).bfloat16().requires_grad_(True)
    w, b = _parameter(torch.randn(N, 64, device=DEV, generator=g)), _parameter(torch.randn(N, device=DEV, generator=g))
    dy = torch.randn(M, N + (8 if strided else 0), device=DEV, generator=g).bfloat16()[:, :N]
    ops.linear(x, w, b).backward(dy)
    assert w.told == 1 and b.told == 0 and not b.main_grad.any()
    want = dy.double().sum(0)
    # fp32 sums of M values of order one, rounded to 16 bits once
    assert float(((b.grad.double() - want).abs() - 2.0 ** -8 * want.abs()).max()) < 2.0 ** -20 * M ** 0.5 * 8


@pytest.mark.parametrize("T,H", [(1, 8), (5, 1536), (700, 1536), (4097, 256), (3000, 8192)])
@pytest.mark.parametrize("residual,gemma", [(False, False), (True, True)])
def test_norm_weight_values(T, H, residual, gemma):
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
    assert torch.equal(*dx) and torch.equal(w.grad, plain.grad) and w.told == 0 and not w.main_grad.any()
    s = x.detach().double() if r is None else (x.detach().float() + r.detach().float()).bfloat16().double()
    want = (dy.double() * s * torch.rsqrt(s.pow(2).mean(-1, keepdim=True) + 1e-6)).sum(0)
    assert float(((w.grad.double() - want).abs() - 2.0 ** -8 * want.abs()).max()) < 2.0 ** -20 * (4.0 + T ** 0.5 * 8)
