"""Weight gradients over few tokens (tiles of 128 x 128): around the edges of a stage of 32 tokens, few and many tiles, experts."""
import sys

import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.ops import _lib as L, train_gemm as tg

G = sys.modules["areal_vllm_amd.ops.grouped_gemm"]
DEV = "cuda:0"
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 31, 32, 33, 65, 256, 287, 700])
@pytest.mark.parametrize("N,K", [(128, 128), (1152, 384), (4096, 4096)])
def test_dense(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M + N)
    # what lies past the last token and beside the columns must not be read: operands and gradient are cut out of larger ones
    dy, x = torch.full((M + 40, N + 8), float("nan"), device=DEV).bfloat16(), torch.full((M + 40, K + 8), float("inf"), device=DEV).bfloat16()
    dy[:M, :N] = torch.randn(M, N, device=DEV, generator=g).bfloat16()
    x[:M, :K] = torch.randn(M, K, device=DEV, generator=g).bfloat16()
    dy, x = dy[:M, :N], x[:M, :K]
    whole = torch.randn(N, K + 1, device=DEV, generator=g)
    want = whole.double()
    want[:, :K] += dy.double().t() @ x.double()
    L.check(L.lib().areal_tgemm_wgrad_few(L.ptr(dy), L.c_int64(N + 8), L.ptr(x), L.c_int64(K + 8), L.ptr(whole), L.c_int64(K + 1),
                                          L.c_int(M), L.c_int(N), L.c_int(K), L.stream_ptr()), "tgemm_wgrad_few")
    # fp32 sums of M products of size one
    assert float((whole.double() - want).abs().max()) < 1e-3 * max(1.0, M ** 0.5 / 16)
    assert torch.equal(whole[:, K].double(), want[:, K])


@pytest.mark.parametrize("counts", [[0, 1, 255, 256, 257, 0, 700, 300], [5000], [3000] + [100] * 23, [31, 32, 33, 0]])
@pytest.mark.parametrize("N,K", [(128, 128), (256, 512), (1536, 768)])
@pytest.mark.parametrize("form", ["by expert", "over all XCDs", "large"])
def test_grouped(counts, N, K, form, monkeypatch):
    monkeypatch.setenv("AREAL_GROUPED_GEMM", "hip")
    monkeypatch.delenv("AREAL_GROUPED_GEMM_TILE_M", raising=False)
    if form == "large" and K % 256:
        pytest.skip("tiles of 256 columns")
    monkeypatch.setattr(G, "FEW_WGRAD_ROWS", 0)
    monkeypatch.setattr(G, "_big_wgrad", lambda *a: form == "large")
    monkeypatch.setattr(G, "_spread_experts", lambda *a: form == "over all XCDs")
    E, T = len(counts), sum(counts)
    g = torch.Generator(device=DEV).manual_seed(T + N + K)
    x = torch.randn(T, K, device=DEV, generator=g).bfloat16()
    w = (torch.randn(E, N, K, device=DEV, generator=g) / K ** 0.5).bfloat16().requires_grad_(True)
    w.main_grad = torch.ones(E, N, K, device=DEV)
    dy = (torch.randn(T, N, device=DEV, generator=g) / N ** 0.5).bfloat16()
    ops.grouped_gemm(x, w, counts).backward(dy)
    at = 0
    for e, n in enumerate(counts):
        want = dy[at:at + n].double().t() @ x[at:at + n].double()
        # fp32 sums of up to 5000 products of size N ** -0.5
        assert float((w.main_grad[e].double() - 1.0 - want).abs().max()) < 1e-4
        at += n


def test_rule_takes_both():
    assert tg._wgrad_few(700, 192) and tg._wgrad_few(1500, 1680) and tg._wgrad_few(1024, 14244)
    assert not tg._wgrad_few(32768, 192) and not tg._wgrad_few(700, 840) and not tg._wgrad_few(1500, 14244)


@pytest.mark.parametrize("M,N,K", [(700, 512, 512), (1024, 512, 512), (1500, 2048, 1536), (2048, 1536, 1536), (700, 2048, 1536), (1031, 6144, 2048)])
def test_no_less_precise_than_large_tiles(M, N, K):
    """The chosen form's error against 64 bits beside that of the large tiles with the parts that they would take."""
    g = torch.Generator(device=DEV).manual_seed(M + N)
    dy, x = torch.randn(M, N, device=DEV, generator=g).bfloat16(), torch.randn(M, K, device=DEV, generator=g).bfloat16()
    want = dy.double().t() @ x.double()
    parts = tg._tile_plan(-(-M // 128), -(-N // 256) * (K // 256), 5)[2]
    err = [float((tg.tgemm_wgrad_(torch.zeros(N, K, device=DEV), dy, x, splits=s).double() - want).norm() / want.norm()) for s in (parts, 0)]
    assert err[1] <= 1.02 * err[0], err  # (the mean over a quarter of a million roundings and more)


@pytest.mark.parametrize("splits", [0, 1, 2])
def test_large_gradients_are_streamed(splits):
    """Gradients from 2^26 elements on pass the caches by: the large tiles' other form."""
    M, N, K = 1700, 65536 + 128, 1024
    assert not tg._wgrad_few(M, N // 128 * (K // 128))
    g = torch.Generator(device=DEV).manual_seed(splits)
    dy, x = torch.randn(M, N, device=DEV, generator=g).bfloat16(), torch.randn(M, K, device=DEV, generator=g).bfloat16()
    whole = torch.randn(N, K + 1, device=DEV, generator=g)
    before = whole.clone()
    tg.tgemm_wgrad_(whole[:, :K], dy, x, splits=splits)
    for lo, hi in ((0, 300), (32700, 33100), (N - 400, N)):
        want = before[lo:hi, :K].double() + dy[:, lo:hi].double().t() @ x.double()
        # fp32 sums of 1700 products of size one
        assert float((whole[lo:hi, :K].double() - want).abs().max()) < 1e-3 * M ** 0.5 / 16
    assert torch.equal(whole[:, K], before[:, K])


def test_large_grouped_gradients_are_streamed(monkeypatch):
    monkeypatch.setenv("AREAL_GROUPED_GEMM", "hip")
    monkeypatch.delenv("AREAL_GROUPED_GEMM_TILE_M", raising=False)
    monkeypatch.setattr(G, "FEW_WGRAD_ROWS", 0)
    monkeypatch.setattr(G, "_big_wgrad", lambda *a: True)
    counts, N, K = [0, 1, 300, 257, 64, 0, 700, 129], 4096 + 128, 2048
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn(sum(counts), K, device=DEV, generator=g).bfloat16()
    w = torch.empty(len(counts), N, K, device=DEV, dtype=torch.bfloat16).normal_(0, K ** -0.5, generator=g).requires_grad_(True)
    w.main_grad = torch.ones(len(counts), N, K, device=DEV)
    assert w.numel() >= 1 << 26
    dy = (torch.randn(sum(counts), N, device=DEV, generator=g) / N ** 0.5).bfloat16()
    ops.grouped_gemm(x, w, counts).backward(dy)
    at = 0
    for e, n in enumerate(counts):
        want = dy[at:at + n].double().t() @ x[at:at + n].double()
        # fp32 sums of up to 700 products of size N ** -0.5
        assert float((w.main_grad[e].double() - 1.0 - want).abs().max()) < 1e-4
        at += n
