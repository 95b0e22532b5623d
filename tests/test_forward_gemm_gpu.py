"""y = x W^T with the tiles beyond full rounds split over the reduction: ragged rows, widths that end inside a tile."""
import pytest
import torch

from areal_vllm_amd.ops import train_gemm as tg

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


# all tiles in parts; 256 whole ones and the rest in parts
@pytest.mark.parametrize("M,K,N,plan", [(257, 1664, 264, (0, 13)), (700, 896, 1536, (0, 4)), (1, 256, 12, (0, 2)),
                                        (4353, 640, 3848, (256, 3)), (300, 384, 1000, (0, 3))])
def test_parts(M, K, N, plan):
    g = torch.Generator(device=DEV).manual_seed(M + K)
    x = torch.full((M + 256, K + 8), float("nan"), device=DEV).bfloat16()[:M, :K]
    w = torch.full((N + 256, K + 8), float("nan"), device=DEV).bfloat16()[:N, :K]
    x.copy_(torch.randn(M, K, device=DEV, generator=g))
    w.copy_(torch.randn(N, K, device=DEV, generator=g) / K ** 0.5)
    out = torch.full((M, N + 8), 7.0, device=DEV).bfloat16()
    got = tg.tgemm_tn(x, w, out=out[:, :N], plan=plan)
    want = x.double() @ w.double().t()
    # outputs of size one (up to 6), rounded to bf16 once: 2^-9 relative; the fp32 sums are far more accurate
    assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())
    assert bool((out[:, N:] == 7.0).all())


@pytest.mark.parametrize("M,K,N,own", [(700, 8960, 1536, True), (700, 1536, 17920, False), (8192, 1536, 151936, True),
                                       (300, 1536, 151936, False), (6000, 18944, 3584, True), (20000, 18944, 3584, False),
                                       (1999, 11008, 4096, True), (701, 16384, 64, True), (601, 128, 98304 + 8, True)])
def test_rule(M, K, N, own):
    assert tg._forward_own(M, K, N) == own
    g = torch.Generator(device=DEV).manual_seed(M + K)
    x = torch.randn(M, K, device=DEV, generator=g).bfloat16()
    w = (torch.randn(N, K, device=DEV, generator=g) / K ** 0.5).bfloat16()
    got = tg.forward(x, w)
    assert got.shape == (M, N)
    rows = torch.cat([torch.arange(0, M, max(1, M // 500), device=DEV), torch.arange(max(0, M - 300), M, device=DEV)])
    for at in range(0, N, 16384):  # (float64: some rows of every tile, and all of the ragged last one)
        want = x[rows].double() @ w[at:at + 16384].double().t()
        assert bool(((got[rows, at:at + 16384].double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())  # as above
