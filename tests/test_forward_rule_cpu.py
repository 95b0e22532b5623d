"""Which products of a forward pass go to the own kernel: sizes at which the library was measured ahead do not."""
import pytest

from areal_vllm_amd.ops import train_gemm as tg


@pytest.mark.parametrize("M,K,N,own", [
    (2048, 8960, 5120, False), (1100, 11008, 8192, False), (800, 8960, 512, False), (800, 8192, 1536, False),  # few rows: up to 19 %
    (9000, 18944, 3584, False), (2048, 18944, 5120, False), (6000, 16384, 8192, False),  # full rounds; one of 160 tiles
    (4500, 18944, 4096, True), (9000, 18944, 5120, True), (300, 18944, 3584, True), (256, 18944, 3584, False),
    (1500, 8960, 1536, True), (2500, 8960, 1536, False), (12288, 28672, 1536, True), (12289, 28672, 1536, False),
])
def test_deep(M, K, N, own):
    assert tg._forward_own(M, K, N) == own


@pytest.mark.parametrize("M,K,N,written,reduced", [
    (1642, 4096, 65536, False, False), (1642, 2048, 65536, False, True), (8192, 1536, 151936, True, True),
    (8192, 4096, 151936, False, False), (4000, 4096, 151936, False, True), (8192, 5120, 151936, True, True), (599, 1536, 151936, False, False),
])
def test_vocabulary(M, K, N, written, reduced):
    assert tg._forward_own(M, K, N) == written and tg._stats_own(M, K, N) == reduced


@pytest.mark.parametrize("M,R,C,own", [(2, 28672, 2048, True), (10000, 8192, 1024, False), (3000, 28672, 4096, False),
                                       (3000, 37888, 3584, True), (32768, 17920, 1536, True), (700, 1536, 8960, False),
                                       (12000, 1536, 8960, True)])
def test_input_gradients(M, R, C, own):
    assert tg._dgrad_own(M, R, C) == own


def test_few_rows_take_more_parts():
    assert tg.dgrad_cost(2, 17920, 1536)[2] == 35 and tg.dgrad_cost(256, 17920, 1536)[2] == 28
