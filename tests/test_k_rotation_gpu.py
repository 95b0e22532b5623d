"""Products whose workgroups start their reduction at different steps (weight rows of a multiple of 4096 bytes): every step is
taken once. Sixteenths make every partial sum exact in fp32, so any order has the same bits."""
import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.ops import decode_gemm as dg

pytestmark = pytest.mark.gpu


def _ints(*shape):
    return (torch.randint(-2, 3, shape, device="cuda") / 16).bfloat16()


@pytest.mark.parametrize("M,N,K", [(1, 8192, 2048), (33, 8224, 4096), (64, 8192 + 96, 2048), (65, 9000 // 32 * 32, 6144),
                                   (128, 8192, 14336), (129, 8192, 2048), (64, 8192, 1984), (1, 16384, 2048), (64, 16384 + 96, 4096),
                                   (100, 32768 + 32, 6144), (128, 32768, 2048)])
def test_decode_gemm_takes_every_step_once(M, N, K):
    torch.manual_seed(M)
    x, w = _ints(M, K), _ints(N, K)
    ref = (x.float() @ w.float().t())
    assert torch.equal(dg.dgemm(x, w), ref.bfloat16())
    assert dg.pick_config(M, N, K, dg.EPI_BF16)[2] == 1
    for stages in (2, 3):
        assert torch.equal(dg.dgemm(x, w, cfg=8, stages=stages), ref.bfloat16())
        assert torch.equal(dg.dgemm(x, w, cfg=4, stages=stages, loader_waves=4), ref.bfloat16())  # (rotated where it is wide)


@pytest.mark.parametrize("M,F,K", [(1, 512, 2048), (64, 4096, 4096), (130, 1000, 2048), (200, 1024, 2048),
                                   (1, 8192, 2048), (100, 8192 + 40, 6144), (200, 8192, 2048)])
def test_decode_swiglu_takes_every_step_once(M, F, K):
    torch.manual_seed(F)
    x, w = _ints(M, K), _ints(2 * F, K)
    whole = (x.float() @ w.float().t()).double()
    ref = torch.nn.functional.silu(whole[:, :F]) * whole[:, F:]
    out = dg.dgemm_swiglu_balanced(x, w)
    # roundings to bf16 (half a step: 2^-8 of the value) of gate, up and result; the gate's passes silu with a factor of at most
    # 1 + |gate|
    assert ((out.double() - ref).abs() <= ref.abs() * (3 + whole[:, :F].abs()) * 2.0 ** -8 + 1e-6).all()


@pytest.mark.parametrize("T,k,E,F,K", [(1, 1, 4, 64, 2048), (40, 8, 128, 64, 2048), (66, 2, 4, 128, 4096), (300, 2, 4, 64, 2048),
                                         (11, 8, 128, 192, 2048)])
def test_grouped_gemm_takes_every_step_once(T, k, E, F, K):
    torch.manual_seed(T)
    x, w = _ints(T, K), _ints(E, 2 * F, K)
    topi = torch.rand(T, E, device="cuda").topk(k, -1).indices.reshape(-1)
    order, inv, src_row, offsets = ops.moe_sort(topi, E, k)
    xs = ops.moe_permute(x, order, inv, k, src_row)
    out = ops.grouped_gemm_offsets(xs, w, offsets[:E + 1])
    ref = torch.einsum("tk,tnk->tn", xs.float().cpu(), w.float().cpu()[topi[order].cpu()])
    assert torch.equal(out.cpu(), ref.bfloat16())
    assert torch.equal(ops.grouped_gate_up(x, src_row, w, offsets[:E + 1]), ops.swiglu(out))


@pytest.mark.parametrize("T,k,E,F,K", [(64, 8, 128, 192, 2048), (70, 2, 8, 2176, 4096)])
def test_a_row_has_the_same_bits_whatever_the_others_choose(T, k, E, F, K):
    torch.manual_seed(T)
    x = torch.randn(T, K, device="cuda").bfloat16()
    w = (torch.randn(E, 2 * F, K, device="cuda") * K ** -0.5).bfloat16()
    topi = torch.rand(T, E, device="cuda").topk(k, -1).indices
    crowded = topi.clone()
    crowded[5:] = torch.arange(k, device="cuda")  # several row tiles an expert ahead of the first five rows' experts
    rows = []
    for choice in (topi, crowded):
        order, inv, src_row, offsets = ops.moe_sort(choice.reshape(-1), E, k)
        first = inv.view(T, k)[:5].reshape(-1)
        xs = ops.moe_permute(x, order, inv, k, src_row)
        rows.append((ops.grouped_gemm_offsets(xs, w, offsets[:E + 1])[first], ops.grouped_gate_up(x, src_row, w, offsets[:E + 1])[first]))
    for a, b in zip(*rows):
        assert torch.equal(a, b)
