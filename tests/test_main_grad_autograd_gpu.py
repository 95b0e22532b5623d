"""Gradients of biases and norm weights go through autograd, also where an fp32 buffer stands behind the parameter: what hangs on the
parameter sees them, and one backward pass reports each once."""
import pytest
import torch

from areal_vllm_amd import ops

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
