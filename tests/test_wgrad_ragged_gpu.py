"""Weight gradients whose token count is no multiple of a tile."""
import pytest
import torch

from areal_vllm_amd.ops import train_gemm as tg

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [256, 257, 319, 320, 383, 700, 1023, 2049, 8191])
@pytest.mark.parametrize("N,K", [(128, 256), (384, 512), (2048, 1536)])
@pytest.mark.parametrize("splits", [0, 1, 2])
def test_ragged_token_counts(M, N, K, splits):
    g = torch.Generator(device=DEV).manual_seed(M + N)
    # rows past the last token hold what must not be read: the operands are cut out of larger ones
    dy = torch.full((M + 130, N + 8), float("nan"), device=DEV).bfloat16()
    x = torch.full((M + 130, K + 8), float("inf"), device=DEV).bfloat16()
    dy[:M, :N] = torch.randn(M, N, device=DEV, generator=g).bfloat16()
    x[:M, :K] = torch.randn(M, K, device=DEV, generator=g).bfloat16()
    dy, x = dy[:M, :N], x[:M, :K]
    base = torch.randn(N, K, device=DEV, generator=g)
    assert tg.wgrad_supported(dy, x, base)
    got = tg.tgemm_wgrad_(base.clone(), dy, x, splits=splits)
    want = base.double() + dy.double().t() @ x.double()
    # fp32 sums of M products of size one: 2^-24 sqrt(M) relative per addition, far below 1e-3
    assert float((got.double() - want).abs().max()) < 1e-3 * max(1.0, M ** 0.5 / 16)


@pytest.mark.parametrize("M,N,K", [(256, 128, 256), (700, 384, 512)])
@pytest.mark.parametrize("which", ["dy", "x", "overlapping"])
def test_rows_that_repeat(M, N, K, which):
    """An output gradient that is the same for all rows (of a mean over them), an input broadcast over them, rows that overlap."""
    from areal_vllm_amd.ops.linear import _accumulate_wgrad

    g = torch.Generator(device=DEV).manual_seed(M)
    dy, x = (torch.randn(M, n, device=DEV, generator=g).bfloat16() for n in (N, K))
    if which == "dy":
        dy = dy[:1].expand(M, N)
    elif which == "x":
        x = x[:1].expand(M, K)
    else:
        dy = torch.randn(M * 64 + N, device=DEV, generator=g).bfloat16().as_strided((M, N), (64, 1))
    w = torch.nn.Parameter(torch.zeros(N, K, device=DEV).bfloat16())
    w.main_grad = torch.zeros(N, K, device=DEV)
    _accumulate_wgrad(w, dy, x)
    want = dy.double().contiguous().t() @ x.double().contiguous()
    # fp32 sums of M products of size one, the same M times over where rows repeat
    assert float((w.main_grad.double() - want).abs().max()) < 1e-5 * M
