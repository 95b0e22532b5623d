"""Input-gradient GEMM dX = dY . W from the weight as it lies: ragged row counts, one and several parts of the reduction."""
import pytest
import torch

from areal_vllm_amd.ops import train_gemm as tg

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 63, 64, 129, 255, 256, 257, 700, 1024])
@pytest.mark.parametrize("R,C", [(128, 256), (384, 512), (1536, 1280), (17920, 256)])
@pytest.mark.parametrize("splits", [0, 1, 2])
def test_dgrad(M, R, C, splits):
    g = torch.Generator(device=DEV).manual_seed(M + R)
    # rows past the last one, and what lies beside the operands, must not be read
    dy = torch.full((M + 256, R + 8), float("nan"), device=DEV).bfloat16()
    w = torch.full((R + 64, C + 16), float("nan"), device=DEV).bfloat16()
    dy[:M, :R] = torch.randn(M, R, device=DEV, generator=g).bfloat16()
    w[:R, :C] = (torch.randn(R, C, device=DEV, generator=g) / R ** 0.5).bfloat16()
    dy, w = dy[:M, :R], w[:R, :C]
    assert tg.dgrad_supported(dy, w)
    if splits == 2 and R == 128:
        pytest.skip("one pair of the reduction cannot be split")
    got = tg.tgemm_nn(dy, w, splits=splits)
    want = dy.double() @ w.double()
    # outputs of size one (up to 6), rounded to bf16 once: 2^-9 relative; the fp32 sums are far more accurate
    assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())


# full rounds of whole tiles, then the rest in parts: 264 tiles in 6 parts, 258 of 13 pairs, 520 with a ragged last row of tiles
@pytest.mark.parametrize("M,R,C,plan", [(16641, 1536, 1024, (256, 6)), (256 * 43, 1664, 1536, (256, 13)), (33025, 384, 1024, (520, 1))])
def test_whole_tiles_and_parts(M, R, C, plan):
    g = torch.Generator(device=DEV).manual_seed(M)
    dy = torch.full((M + 256, R + 8), float("nan"), device=DEV).bfloat16()[:M, :R]
    w = torch.full((R + 64, C + 16), float("nan"), device=DEV).bfloat16()[:R, :C]
    dy.copy_(torch.randn(M, R, device=DEV, generator=g))
    w.copy_(torch.randn(R, C, device=DEV, generator=g) / R ** 0.5)
    assert tg.dgrad_cost(M, R, C)[1:] == plan
    got = tg.tgemm_nn(dy, w)
    want = dy.double() @ w.double()
    assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())  # one rounding, as above
    assert torch.equal(got, tg.tgemm_nn(dy, w))


def test_parts_have_work():
    for M in (1, 256, 700, 4096, 30000):
        for R in (128, 256, 1536, 17920, 151936):
            for C in (256, 1536, 8960):
                s = tg.dgrad_cost(M, R, C)[2]
                pairs = R // 128
                assert 1 <= s <= pairs and -(-pairs // -(-pairs // s)) == s


@pytest.mark.parametrize("M", [1, 17, 200])
def test_parts_hold_the_rows_that_there_are(M):
    R, C, splits = 1536, 512, 4
    dy, w = torch.randn(M, R, device=DEV).bfloat16(), torch.randn(R, C, device=DEV).bfloat16()
    out = torch.empty(M, C, device=DEV, dtype=torch.bfloat16)
    part = torch.full((splits, 2, 256, 256), 7.0, device=DEV)
    tg.L.check(tg.L.lib().areal_tgemm_nn(tg.L.ptr(dy), tg.L.c_int64(R), tg.L.ptr(w), tg.L.c_int64(C), tg.L.ptr(out), tg.L.c_int64(C),
                                         tg.L.ptr(part), tg.L.c_int(0), tg.L.c_int(splits), tg.L.c_int(M), tg.L.c_int(R),
                                         tg.L.c_int(C), tg.L.stream_ptr()), "tgemm_nn")
    assert bool((part[:, :, M:] == 7.0).all())  # a few rows' parts are a few rows: the others are most of the call's bytes
    assert torch.equal(out, part[:, :, :M].sum(0).permute(1, 0, 2).reshape(M, C).bfloat16())  # (four parts: added in order)
