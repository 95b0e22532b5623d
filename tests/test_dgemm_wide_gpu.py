"""The product for wide outputs, whose workgroups walk several column ranges each, against double precision."""
import pytest
import torch

from areal_vllm_amd.ops import decode_gemm as dg

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# one step and fewer than the ring has stages, rows that start their reduction apart (2048, 4096), ranges of 64 (one a workgroup, last
# one short) to 160 columns, a last round of few
@pytest.mark.parametrize("M", [65, 96, 97, 128, 129, 160])
@pytest.mark.parametrize("N,K", [(16384, 64), (20004, 128), (40960, 320), (40964, 192), (100352, 2048), (151936, 896), (16388, 4096)])
def test_against_double_precision(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x = torch.randn(M + 1, K + 8, device=DEV, generator=g).bfloat16()[:M, :K]  # rows further apart than they are long
    w = (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).bfloat16()
    assert dg.serves_wide(x, w)
    got = dg.dgemm_wide(x, w)
    want = x.double() @ w.double().t()
    # rounded once, and a sum next to a rounding edge to the other side of it: half a step is 2^-9, fp32 sums of terms of order one 2^-17
    assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -17).all()
    assert float((got != want.bfloat16()).double().mean()) < 1e-3 and torch.equal(got, dg.dgemm_wide(x, w))


def test_what_it_does_not_take():
    x, w = torch.randn(65, 128, device=DEV).bfloat16(), torch.randn(16384, 128, device=DEV).bfloat16()
    half = w[:, :64].contiguous()
    assert dg.serves_wide(x, w) and not dg.serves_wide(x, w[:16380]) and dg.takes_wide(x, w[:16380]) and not dg.takes_wide(x, w[:16382])
    assert not dg.takes_wide(x.float(), w) and not dg.takes_wide(x[:, ::2], half) and not dg.takes_wide(x[:, 4:68], half)
    assert not dg.takes_wide(x[:64], w) and not dg.takes_wide(torch.randn(161, 128, device=DEV).bfloat16(), w)


@pytest.mark.parametrize("depth", [64, 192])
def test_weights_of_another_depth_are_refused(depth):
    """The kernel steps through the weight in rows as deep as x: on the host, before anything is launched."""
    x, w = torch.randn(65, 128, device=DEV).bfloat16(), torch.randn(16384, depth, device=DEV).bfloat16()
    assert not dg.takes_wide(x, w) and not dg.serves_wide(x, w) and not dg.takes_wide(x, w.view(-1))
    with pytest.raises(AssertionError):
        dg.dgemm_wide(x, w)
