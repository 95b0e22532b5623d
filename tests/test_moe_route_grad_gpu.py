"""Gradients of a routed layer's glue: the weights of the choices and the recombination, one launch each."""
import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.ops import moe

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,k", [(1, 1, 1), (3, 2, 2), (5, 63, 7), (4, 64, 64), (1025, 65, 8), (300, 128, 8), (9, 257, 33), (2, 512, 64)])
@pytest.mark.parametrize("norm", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_weights_of_the_choices(T, E, k, norm, dtype):
    g = torch.Generator(device=DEV).manual_seed(T + E)
    z = (torch.randn(T, E, device=DEV, generator=g) * 2).to(dtype).requires_grad_(True)
    v, i = moe.moe_topk_grad(z, k, norm)
    assert v.dtype == torch.float32 and not i.requires_grad
    gv = torch.randn(T, k, device=DEV, generator=g)
    (dz,) = torch.autograd.grad(v, z, gv)
    z64 = z.detach().double().requires_grad_(True)
    want = torch.softmax(z64, -1).gather(1, i)
    want = want / want.sum(-1, keepdim=True) if norm else want
    (d64,) = torch.autograd.grad(want, z64, gv.double())
    # an exponential is off by a few 2^-24, a sum of 512 of them and the quotients by some more; the terms of a gradient cancel
    # down from the size of g p, 16-bit results are rounded once
    assert float((v.double() - want).detach().abs().max()) < 2.0 ** -19
    err = (dz.double() - d64).abs()
    assert float((err - (2.0 ** -8 * d64.abs() if dtype == torch.bfloat16 else 0.0)).max()) < 2.0 ** -18 * max(1.0, float(gv.abs().max()))


@pytest.mark.parametrize("E,k,dtype", [(8, 8, torch.float32), (64, 64, torch.float32), (64, 64, torch.bfloat16), (512, 64, torch.float32)])
def test_small_probabilities_are_as_exact_as_large_ones(E, k, dtype):
    """Logits that are multiples of 1/2 down to -80 below one that is far above all others: differences and sums are exact but for the
    last bits. The exponential is off by a unit in the last place (2^-23), the sum (terms of e^-8 and less beside 1) and the quotient by
    less: below 2^-21 together. The exponential of a rounded product would be off by |logit - max| 2^-24, up to 2^-18."""
    g = torch.Generator(device=DEV).manual_seed(E)
    z = (-8.0 - torch.randint(0, 145, (200, E), device=DEV, generator=g) / 2.0).to(dtype)
    z[:, E // 3] = 0.0
    z.requires_grad_(True)
    v, i = moe.moe_topk_grad(z, k, False)
    z64 = z.detach().double().requires_grad_(True)
    want = torch.softmax(z64, -1).gather(1, i)
    assert float(((v.double() - want) / want).detach().abs().max()) < 2.0 ** -21
    gv = torch.rand(200, k, device=DEV, generator=g) + 0.5
    (dz,) = torch.autograd.grad(v, z, gv)
    (d64,) = torch.autograd.grad(want, z64, gv.double())
    # p (g - sum of p g), the bracket at most 1.5: p's error, and some 2^-24 of the bracket; 16-bit results are rounded once
    err = ((dz.double() - d64).abs() / torch.softmax(z64.detach(), -1)).max()
    assert float(err) < (2.0 ** -20 if dtype == torch.float32 else 2.0 ** -8)


def test_choices_next_to_infinities():
    z = torch.full((2, 70), -float("inf"), device=DEV)
    z[:, 3], z[:, 69] = 1.0, 2.0
    z.requires_grad_(True)
    v, i = moe.moe_topk_grad(z, 2, True)
    assert i.tolist() == [[69, 3]] * 2
    (dz,) = torch.autograd.grad(v, z, torch.tensor([[1.0, 0.0], [0.0, 1.0]], device=DEV))
    p = float(torch.sigmoid(torch.tensor(1.0))) * (1 - float(torch.sigmoid(torch.tensor(1.0))))
    assert torch.allclose(dz[:, 69].cpu(), torch.tensor([p, -p]), atol=1e-6) and torch.allclose(dz[:, 3].cpu(), torch.tensor([-p, p]), atol=1e-6)
    assert int((dz != 0).sum()) == 4


@pytest.mark.parametrize("E,k,finite", [(2, 2, [0]), (70, 5, [0, 69]), (70, 64, [66, 0, 3]), (512, 9, [511]), (64, 64, [0])])
@pytest.mark.parametrize("norm", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_more_choices_than_finite_logits(E, k, finite, norm, dtype):
    """Every choice is another expert, those of weight 0 the first ones that are left, and the gradient is softmax's of these choices."""
    z = torch.full((3, E), -float("inf"), device=DEV)
    z[:, finite] = torch.tensor([[0.5 * j for j in range(len(finite))]] * 3, device=DEV)
    z = z.to(dtype).requires_grad_(True)
    v, i = moe.moe_topk_grad(z, k, norm)
    rest = [e for e in range(E) if e not in finite]
    assert i.tolist() == [(finite[::-1] + rest)[:k]] * 3
    gv = torch.arange(3 * k, device=DEV).view(3, k) / 8.0
    (dz,) = torch.autograd.grad(v, z, gv)
    z64 = z.detach().double().requires_grad_(True)
    want = torch.softmax(z64, -1).gather(1, i)
    want = want / want.sum(-1, keepdim=True) if norm else want
    (d64,) = torch.autograd.grad(want, z64, gv.double())
    assert float((v.double() - want).detach().abs().max()) < 2.0 ** -21  # as of small probabilities
    # terms of up to max(gv), a few 2^-24 each; 16-bit results are rounded once
    top = float(gv.max())
    assert float(((dz.double() - d64).abs() - (2.0 ** -8 * d64.abs() if dtype == torch.bfloat16 else 0.0)).max()) < 2.0 ** -20 * top


@pytest.mark.parametrize("E,k", [(5, 2), (64, 8), (130, 3)])
@pytest.mark.parametrize("norm", [True, False])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), None])
def test_a_row_that_softmax_makes_nan_is_nan(E, k, norm, bad):
    """None: a row of nothing but -inf. Weights and gradients of that row, and of no other; choices that exist."""
    g = torch.Generator(device=DEV).manual_seed(E)
    z = torch.randn(3, E, device=DEV, generator=g)
    z[1] = -float("inf") if bad is None else z[1]
    if bad is not None:
        z[1, E - 2] = bad
    assert bool(torch.softmax(z, -1)[1].isnan().all())
    z.requires_grad_(True)
    v, i = moe.moe_topk_grad(z, k, norm)
    (dz,) = torch.autograd.grad(v, z, torch.ones_like(v) + torch.arange(k, device=DEV))
    for t in (v, dz):
        assert bool(t[1].isnan().all()) and bool(torch.isfinite(t[[0, 2]]).all())
    assert int(i.min()) >= 0 and int(i.max()) < E


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
