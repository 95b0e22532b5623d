"""The launches of a routed-expert layer's decode step that do the work of several: gather + gate|up GEMM + activation, router
partial sums + top-k, recombination + residual + RMSNorm."""
import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.ops import moe as moe_ops

pytestmark = pytest.mark.gpu


def _routed(T, k, E, seed, skew=False):
    g = torch.Generator().manual_seed(seed)
    prob = torch.rand(T, E, generator=g)
    if skew:  # everything on the last experts: the others own no rows
        prob[:, : E - k - 1] = -1.0
    topi = prob.topk(k, -1).indices.reshape(-1).cuda()
    return ops.moe_sort(topi, E, k)


@pytest.mark.parametrize("T,k,E,F,K,skew", [(1, 1, 4, 64, 64, False), (7, 8, 128, 768, 2048, False), (64, 8, 128, 768, 2048, False),
                                            (65, 2, 8, 192, 128, False), (129, 2, 3, 64, 192, True), (500, 4, 16, 320, 1024, True)])
def test_gate_up_in_one_launch_has_the_bits_of_the_three(T, k, E, F, K, skew):
    torch.manual_seed(T)
    x = torch.randn(T, K, device="cuda").bfloat16()
    w = (torch.randn(E, 2 * F, K, device="cuda") * K ** -0.5).bfloat16()
    order, inv, src_row, offsets = _routed(T, k, E, T, skew)
    assert ops.gate_up_rows_ok(T * k, w)
    out = ops.grouped_gate_up(x, src_row, w, offsets[:E + 1])
    gu = ops.grouped_gemm_offsets(ops.moe_permute(x, order, inv, k, src_row), w, offsets[:E + 1])
    assert torch.equal(out, ops.swiglu(gu))
    shifted = torch.empty(T * K + 1, device="cuda", dtype=torch.bfloat16)[1:].view(T, K)  # rows off the 16-byte grid
    shifted.copy_(x)
    assert torch.equal(out, ops.grouped_gate_up(shifted, src_row, w, offsets[:E + 1]))


@pytest.mark.parametrize("T,k,H,gemma", [(1, 1, 8, False), (5, 8, 2048, False), (64, 9, 2056, True), (33, 16, 8192, False)])
def test_combine_with_residual_and_norm(T, k, H, gemma):
    torch.manual_seed(H)
    ys = torch.randn(T * k, H, device="cuda").bfloat16()
    w = torch.rand(T, k, device="cuda").bfloat16()
    inv = torch.randperm(T * k, device="cuda")
    res, nw = torch.randn(T, H, device="cuda").bfloat16(), torch.randn(H, device="cuda").bfloat16()
    y, out = ops.moe_combine_rmsnorm(ys, w, inv, res, nw, 1e-6, gemma)
    mixed = ops.moe_combine(ys, w, inv.argsort(), inv)
    assert torch.equal(out, (mixed.float() + res.float()).bfloat16())
    o = out.double()
    ref = o * torch.rsqrt(o.square().mean(-1, keepdim=True) + 1e-6) * (nw.double() + float(gemma))
    # one rounding to bf16 (7 stored bits: half a step is at most 2^-8 of the value) behind fp32 arithmetic
    assert ((y.double() - ref).abs() <= ref.abs() * (2.0 ** -8 + 2.0 ** -16)).all()


@pytest.mark.parametrize("T,E,H,k", [(1, 32, 64, 32), (64, 128, 2048, 8), (512, 96, 512, 4), (513, 128, 256, 8), (9, 512, 1024, 2),
                                     (3, 40, 64, 5)])
def test_router_partial_sums_give_the_choices_of_the_whole_product(T, E, H, k):
    torch.manual_seed(E)
    # sixteenths and a few bits: every product and sum is exact in fp32 and in bf16's eight bits or rounds once, so the
    # partial sums of any split have one right answer
    x = (torch.randint(-2, 3, (T, H), device="cuda") / 16).bfloat16()
    r = (torch.randint(-2, 3, (E, H), device="cuda") / 16).bfloat16()
    for dtype in (torch.float32, torch.bfloat16):
        topv, topi = ops.moe_route(x, r, k, True, dtype)
        raw = (x.double() @ r.double().t()).bfloat16()
        wv, wi = ops.moe_topk(raw, k, True, dtype)
        assert torch.equal(topi, wi) and torch.equal(topv, wv)
        p = torch.softmax(raw.double(), -1)
        ref = torch.argsort(p, descending=True, stable=True)[:, :k]  # lowest expert first among equals
        assert torch.equal(topi, ref)


@pytest.mark.parametrize("E", [3, 64, 65, 300, 512])
def test_topk_with_infinities_and_ties(E):
    k = min(E, 8)
    z = torch.zeros(4, E)
    z[0, E // 2:] = float("-inf")  # fewer finite entries than k for small E: the missing choices are expert 0 with weight 0
    z[1, 0] = 3.0
    z[2, E - 1] = 3.0
    topv, topi = ops.moe_topk(z.cuda(), k, False)
    n = min(k, E // 2)
    assert topi[0, :n].tolist() == list(range(n)) and topi[0, n:].eq(0).all() and topv[0, n:].eq(0).all()
    assert topi[1].tolist() == list(range(k)) and topi[3].tolist() == list(range(k))
    assert topi[2].tolist() == [E - 1] + list(range(k - 1))
    assert torch.allclose(topv[3].cpu(), torch.full((k,), 1.0 / E))
    assert moe_ops.moe_topk(z.cuda()[:0], k, False)[0].shape == (0, k)
