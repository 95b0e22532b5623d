"""Which tiles routed experts take: the large ones, one a CU, only where they fill most of the chip's rounds."""
import sys

import pytest

from areal_vllm_amd import ops  # noqa: F401

G = sys.modules["areal_vllm_amd.ops.grouped_gemm"]
M = sys.modules["areal_vllm_amd.ops.moe"]


@pytest.mark.parametrize("T,E,N,K,out,dx,dw", [
    (4 * 400, 4, 2048, 768, False, False, False),  # 66 tiles; 25; 96
    (8 * 400, 8, 2816, 512, True, False, False),  # 182 tiles, 33, 176
    (16 * 400, 16, 2048, 768, False, False, False),  # 264 (a second round for 8), 99, 384
    (16 * 1000, 16, 2816, 2048, True, True, False),
    (16 * 1023, 16, 2048, 768, True, True, False),  # gradients of 1024 rows an expert and more
    (16 * 1024, 16, 2048, 768, True, True, True),  # 384
    (4 * 1024, 4, 2048, 768, True, False, False),  # 96 in one round
    (8 * 1024, 8, 2816, 512, True, False, True),  # 176
    (8 * 2047, 8, 28672, 4096, True, True, False),  # large experts
    (8 * 2048, 8, 28672, 4096, True, True, True),
    (128 * 200, 128, 1536, 2048, True, True, False),  # gradients of few rows
    (128 * 1024, 128, 1536, 2048, True, True, True),
    (128 * 127, 128, 1536, 2048, False, False, False),
])
def test_rule(T, E, N, K, out, dx, dw, monkeypatch):
    monkeypatch.delenv("AREAL_GROUPED_GEMM_TILE_M", raising=False)
    got = G._big_tiles(T, E, N), G._big_tiles(T, E, K), G._big_wgrad(T, E, N, K, [2 * T // E])
    monkeypatch.setenv("AREAL_GROUPED_GEMM_TILE_M", "64")
    assert not G._big_tiles(T, E, N) and not G._big_wgrad(T, E, N, K, [2 * T // E])
    assert got == (out, dx, dw)
    monkeypatch.delenv("AREAL_GROUPED_GEMM_TILE_M")
    assert not G._big_wgrad(T, E, N, K, [9 * T // E])  # behind a crowded expert


@pytest.mark.parametrize("E,N,K,rows,crowd,spread", [  # `crowd`: the largest expert's rows, of the mean's
    (128, 1536, 2048, 500, 1, False), (128, 1536, 2048, 500, 2.9, False), (128, 1536, 2048, 500, 3.1, True),  # 192 tiles
    (128, 2048, 768, 500, 5.9, False), (128, 2048, 768, 500, 6.1, True),  # 96
    (8, 4096, 14336, 500, 2.9, False), (8, 4096, 14336, 500, 3.1, True),  # 3584: 1.5 from 1024 tiles on
    (32, 1024, 1024, 500, 15, False), (32, 1024, 1024, 500, 17, True),  # 64: only behind an expert with more than half of all rows
    (16, 1536, 768, 16, 8, False), (16, 1536, 768, 16, 8.1, True),  # 72
])
def test_spread(E, N, K, rows, crowd, spread):
    most, T = int(rows * crowd), rows * E
    if N // 128 * (K // 128) >= 1024:
        most = int(rows * crowd / 2)
    counts = [(T - most) // (E - 1)] * E
    counts[E // 2] = most
    counts[0] += T - sum(counts)
    assert max(counts) == most and G._spread_experts(T, E, N, K, counts) == spread


@pytest.mark.parametrize("T,E,H,parts", [(64, 128, 2048, True), (512, 128, 2048, True), (128, 128, 4096, True),
                                         (129, 128, 4096, False), (16, 128, 7168, False), (1, 256, 1024, False),
                                         (512, 32, 7168, True), (513, 32, 1024, False), (0, 32, 1024, False)])
def test_router(T, E, H, parts):
    assert M._route_in_parts(T, E, H) == parts
