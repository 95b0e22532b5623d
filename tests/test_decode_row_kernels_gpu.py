"""Row kernels behind a split reduction with the number of slabs known to the compiler, at the edges of their ranges."""
import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.ops import decode_gemm as dg
from areal_vllm_amd.ops import decode_skinny as sk

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [1, 2, 3, 4, 5, 7, 8, 13, 23, 24, 25])
@pytest.mark.parametrize("M,N", [(1, 4), (3, 1020), (2, 1024), (5, 1028), (24, 1536), (7, 1540), (2, 2048), (2, 2052)])
@pytest.mark.parametrize("gemma", [False, True])
def test_residual_and_norm_of_known_slabs(S, M, N, gemma):
    """A bias of zeros takes the kernel that counts the slabs at run time: the same sums in the same order, bit for bit (but for the
    square sum's order where a row is more than one chunk a thread)."""
    g = torch.Generator(device=DEV).manual_seed(S * 100 + N)
    slab = torch.randn(S, M, N, device=DEV, generator=g)
    res = torch.randn(M, N, device=DEV, generator=g).bfloat16()
    w = torch.randn(N, device=DEV, generator=g).bfloat16()
    y, r = dg.splitk_residual_rmsnorm(slab, S, M, N, residual=res, weight=w, gemma=gemma)
    y0, r0 = dg.splitk_residual_rmsnorm(slab, S, M, N, bias=torch.zeros(N, device=DEV).bfloat16(), residual=res, weight=w, gemma=gemma)
    assert torch.equal(r, r0) and torch.equal(y, y0)
    want = slab.double().sum(0).float().bfloat16().double() + res.double()
    # a sum of up to 25 unit normals is off by less than 25 steps of 2^-21 before it is rounded to 8 bits, a few times near an edge
    assert float(((r.double() - want).abs() - 2.0 ** -7 * want.abs()).max()) < 2.0 ** -5


@pytest.mark.parametrize("S", [1, 2, 3, 5, 8, 9])
@pytest.mark.parametrize("T", [1, 160, 161, 700])
@pytest.mark.parametrize("Hq,Hkv,D,bias,rope", [(12, 2, 128, True, True), (3, 1, 128, False, False), (32, 4, 128, False, True), (6, 2, 64, True, True),
                                                (2, 1, 16, False, True)])
def test_rope_and_cache_of_known_slabs(S, T, Hq, Hkv, D, bias, rope):
    """Sums of sixteenths are exact in any order: the same numbers as the separate rotation and cache write, up to the rotation's
    own rounding (its product of one pair is rounded by itself: one step of a value below 8 is 2^-5)."""
    g = torch.Generator(device=DEV).manual_seed(S * 1000 + T + D)
    N = (Hq + 2 * Hkv) * D
    slab = torch.randint(-8, 9, (S, T, N), device=DEV, generator=g).float() / 16
    b = (torch.randint(-8, 9, (N,), device=DEV, generator=g).float() / 16).bfloat16() if bias else None
    pos = torch.randint(0, 500, (T,), device=DEV, generator=g, dtype=torch.int32)
    slots = torch.randperm(32 * 32, device=DEV, generator=g)[:T].long()
    slots[T // 2] = -1
    tab = ops.RotaryTable(D, 512, 1e4, DEV)
    caches = [ops.alloc_kv_cache(32, Hkv, D, torch.bfloat16, DEV) for _ in range(2)]
    q = dg.splitk_rope_cache_write(slab, S, b, pos, slots, tab, *caches[0], Hq, Hkv, D, do_rope=rope)
    want = (slab.sum(0) + (b.float() if bias else 0.0)).bfloat16().view(T, Hq + 2 * Hkv, D).contiguous()
    ops.rope_and_cache_write_(want, pos, slots, tab, *caches[1], Hq, Hkv, rope)
    for got, ref in zip((q, *caches[0]), (want[:, :Hq], *caches[1])):
        assert float((got.double() - ref.double()).abs().max()) <= (2.0 ** -5 if rope else 0.0)
    assert torch.equal(caches[0][1], caches[1][1])  # V is not rotated


@pytest.mark.parametrize("Hq,Hkv,D", [(1, 1, 48), (5, 2, 16), (1, 1, 112)])  # column blocks: no multiple of the 8 XCDs, one or three a head
@pytest.mark.parametrize("M,rt", [(1, 1), (16, 1), (33, 2)])
def test_qkv_rows_of_odd_column_blocks(Hq, Hkv, D, M, rt):
    g = torch.Generator(device=DEV).manual_seed(D + M)
    sixteenths = lambda *shape: torch.randint(-4, 5, shape, device=DEV, generator=g).float() / 16
    N, K = (Hq + 2 * Hkv) * D, 128
    x, w, b = sixteenths(M, K).bfloat16(), sixteenths(N, K).bfloat16(), sixteenths(N).bfloat16()
    pos, slots = torch.zeros(M, device=DEV, dtype=torch.int32), torch.arange(M, device=DEV)
    tab = ops.RotaryTable(D, 4, 1e4, DEV)
    kc, vc = ops.alloc_kv_cache(3, Hkv, D, torch.bfloat16, DEV)
    y = (x.float() @ w.float().t() + b.float()).bfloat16().view(M, Hq + 2 * Hkv, D)
    for rope in (False, True):  # position 0: nothing turns
        kc.zero_(), vc.zero_()
        q = sk.qkv_rope(x, w, b, pos, slots, tab, kc, vc, Hq, Hkv, D, rt, do_rope=rope)
        assert torch.equal(q, y[:, :Hq])
        assert torch.equal(kc[slots // 32, :, slots % 32], y[:, Hq:Hq + Hkv])
        assert torch.equal(vc[slots // 32, :, :, slots % 32], y[:, Hq + Hkv:])


def test_qkv_rows_of_more_rows_than_a_grid_has():
    Hq, Hkv, D, K, M = 1, 1, 16, 64, 65535 * 16 + 17
    g = torch.Generator(device=DEV).manual_seed(1)
    x = (torch.randint(-4, 5, (M, K), device=DEV, generator=g).float() / 16).bfloat16()
    w = (torch.randint(-4, 5, (3 * D, K), device=DEV, generator=g).float() / 16).bfloat16()
    slots = torch.full((M,), -1, device=DEV)
    slots[-1] = 7
    kc, vc = ops.alloc_kv_cache(1, Hkv, D, torch.bfloat16, DEV)
    q = sk.qkv_rope(x, w, None, torch.zeros(M, device=DEV, dtype=torch.int32), slots, ops.RotaryTable(D, 4, 1e4, DEV), kc, vc, Hq, Hkv, D, 1)
    y = (x.float() @ w.float().t()).bfloat16()
    assert torch.equal(q.view(M, D), y[:, :D]) and torch.equal(kc[0, 0, 7], y[-1, D:2 * D]) and torch.equal(vc[0, 0, :, 7], y[-1, 2 * D:])
