"""Grouped GEMM on tiles of 256 x 256: experts without rows, with one, around the edges of a tile, over several tiles."""
import sys

import pytest
import torch

from areal_vllm_amd import ops

G = sys.modules["areal_vllm_amd.ops.grouped_gemm"]
DEV = "cuda:0"
pytestmark = pytest.mark.gpu

COUNTS = [[0, 1, 255, 256, 257, 0, 700, 300], [5000], [0, 0, 130, 127, 900, 129], [200] * 300, [3000] + [100] * 23]


@pytest.mark.parametrize("counts", COUNTS)
@pytest.mark.parametrize("N,K", [(192, 128), (256, 256), (384, 512), (1536, 768)])
def test_big_tiles(counts, N, K, monkeypatch):
    monkeypatch.setenv("AREAL_GROUPED_GEMM", "hip")
    monkeypatch.delenv("AREAL_GROUPED_GEMM_TILE_M", raising=False)
    E, T = len(counts), sum(counts)
    if E * N * K > 1 << 26:
        pytest.skip("one size of many experts is enough")
    monkeypatch.setattr(G, "_big_tiles", lambda *a: True)  # (the rule asks for more tiles)
    monkeypatch.setattr(G, "_big_wgrad", lambda *a: K % 256 == 0 and counts[0] != 3000)  # dW of a crowded expert: small tiles
    g = torch.Generator(device=DEV).manual_seed(T + N + K)
    x = torch.randn(T, K, device=DEV, generator=g).bfloat16().requires_grad_(True)
    w = (torch.randn(E, N, K, device=DEV, generator=g) / K ** 0.5).bfloat16().requires_grad_(True)
    w.main_grad = torch.ones(E, N, K, device=DEV)
    dy = (torch.randn(T, N, device=DEV, generator=g) / N ** 0.5).bfloat16()
    out = ops.grouped_gemm(x, w, counts)
    out.backward(dy)
    at = 0
    for e, n in enumerate(counts):
        xe, we, de = x.detach()[at:at + n].double(), w.detach()[e].double(), dy[at:at + n].double()
        # results of size one, rounded to bf16 once; the fp32 sums are far more accurate
        for got, want in ((out[at:at + n], xe @ we.t()), (x.grad[at:at + n], de @ we)):
            assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())
        if N % 128 == 0 and K % 128 == 0:
            assert float((w.main_grad[e].double() - 1.0 - de.t() @ xe).abs().max()) < 1e-4
        at += n
