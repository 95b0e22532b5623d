"""Decode projections of a few rows against the same arithmetic in fp64 with the same rounding points, and the five-launch
layer inside the runner against the split-K layer."""
import math

import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.ops import decode_skinny as sk

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


def _norm(h, w, gemma):
    x = h.double() * torch.rsqrt(h.double().pow(2).mean(-1, keepdim=True) + 1e-6) * (w.double() + (1.0 if gemma else 0.0))
    return x.bfloat16().double()


def _close(got, want, bits=7):
    # two correctly rounded bf16 values of sums that differ in the last fp32 bits, or products of two such: a few 2^-8
    err = (got.double() - want).abs() - 2.0 ** -bits * want.abs()
    assert float(err.max()) < 2.0 ** -bits * float(want[want != 0].abs().mean()), float(err.max())


@pytest.mark.parametrize("M", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("N,K", [(1536, 1536), (1536, 8960), (3584, 18944), (7, 64), (40, 25600), (300, 576), (5000, 1024)])
def test_linear_residual(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M * 7 + N)
    x = torch.randn(M + 1, K + 8, device=DEV, generator=g).bfloat16()[:M, :K]  # rows further apart than they are long
    w = (torch.randn(N, K, device=DEV, generator=g) / math.sqrt(K)).bfloat16()
    r = torch.randn(M, N, device=DEV, generator=g).bfloat16()
    y = x.double() @ w.double().t()
    _close(sk.linear_residual(x, w), y)
    got = sk.linear_residual(x, w, r)
    _close(got, y.bfloat16().double() + r.double())
    assert torch.equal(got, sk.linear_residual(x, w, r))


@pytest.mark.parametrize("M", [1, 2, 4, 7, 8])
@pytest.mark.parametrize("F,K", [(8960, 1536), (100, 64), (4096, 1024), (11008, 2048), (18944, 3584), (14336, 4096), (36, 8192)])
@pytest.mark.parametrize("gemma,act", [(False, "silu"), (True, "gelu_tanh")])
def test_norm_gated(M, F, K, gemma, act):
    g = torch.Generator(device=DEV).manual_seed(M * 7 + F)
    h = torch.randn(M, K, device=DEV, generator=g).bfloat16() * 3
    nw = torch.rand(K, device=DEV, generator=g).bfloat16() + 0.5
    w = (torch.randn(2 * F, K, device=DEV, generator=g) / math.sqrt(K)).bfloat16()
    y = (_norm(h, nw, gemma) @ w.double().t()).bfloat16().double()
    gate = torch.nn.functional.silu(y[:, :F]) if act == "silu" else torch.nn.functional.gelu(y[:, :F], approximate="tanh")
    # gate and up are rounded before they are multiplied: two values next to a rounding edge may each be off by one step
    _close(sk.norm_gated(h, nw, w, eps=1e-6, gemma=gemma, act=act), gate * y[:, F:], bits=6)


@pytest.mark.parametrize("M", [1, 2, 4, 8])
@pytest.mark.parametrize("Hq,Hkv,D,K,fp8", [(12, 2, 128, 1536, False), (12, 2, 128, 1536, True), (28, 4, 128, 3584, False),
                                            (2, 1, 64, 192, False), (8, 1, 256, 2048, True), (3, 3, 16, 64, False)])
@pytest.mark.parametrize("with_bias", [True, False])
def test_norm_qkv_rope(M, Hq, Hkv, D, K, fp8, with_bias):
    g = torch.Generator(device=DEV).manual_seed(M * 7 + K)
    h = torch.randn(M, K, device=DEV, generator=g).bfloat16()
    nw = torch.rand(K, device=DEV, generator=g).bfloat16() + 0.5
    N = (Hq + 2 * Hkv) * D
    w = (torch.randn(N, K, device=DEV, generator=g) / math.sqrt(K)).bfloat16()
    bias = torch.randn(N, device=DEV, generator=g).bfloat16() if with_bias else None
    pos = torch.randint(0, 500, (M,), device=DEV, generator=g, dtype=torch.int32)
    slots = (torch.randperm(40 * 32, device=DEV, generator=g)[:M]).long()
    if M > 1:
        slots[1] = -1  # a retired row: nothing is written
    tab = ops.RotaryTable(D, 512, 1e4, DEV)
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
    caches = [ops.alloc_kv_cache(40, Hkv, D, dt, DEV) for _ in range(2)]
    q = sk.norm_qkv_rope(h, nw, w, bias, pos, slots, tab, *caches[0], Hq, Hkv, D, eps=1e-6)
    y = _norm(h, nw, False) @ w.double().t()
    if with_bias:
        y = y + bias.double()
    want = y.bfloat16().view(M, Hq + 2 * Hkv, D).contiguous()
    ops.rope_and_cache_write_(want, pos, slots, tab, *caches[1], Hq, Hkv)
    # a rotated value holds its partner's rounding too, whatever its own size: one step of values below 8 is 2^-5
    _close(q, want[:, :Hq].double(), bits=5)
    for a, b in zip(*caches):  # fp8: a value next to a rounding edge of 3 bits of mantissa may take the other one
        _close(a.float(), b.float().double(), bits=2 if fp8 else 5)
        assert torch.equal(a.float() != 0, b.float() != 0) or float(((a.float() != 0) != (b.float() != 0)).sum()) < 3
