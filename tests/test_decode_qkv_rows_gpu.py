"""The one-launch q|k|v projection of normalised rows against the same arithmetic in fp64 with the same rounding points."""
import math

import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.ops import decode_skinny as sk

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


def _close(got, want, bits):
    err = (got.double() - want).abs() - 2.0 ** -bits * want.abs()
    assert float(err.max()) < 2.0 ** -bits * float(want[want != 0].abs().mean()), float(err.max())


@pytest.mark.parametrize("M,row_tiles", [(1, 1), (7, 1), (16, 1), (17, 1), (24, 1), (24, 2), (32, 2), (33, 1), (33, 2), (100, 2)])
@pytest.mark.parametrize("Hq,Hkv,D,K,fp8,bias", [(12, 2, 128, 1536, False, True), (12, 2, 128, 1536, True, True), (8, 1, 256, 2304, True, False),
                                                 (2, 1, 64, 192, False, True), (3, 3, 16, 64, False, False), (4, 4, 64, 576, False, True),
                                                 (1, 1, 128, 5120, False, True)])  # deeper than two sets of registers
def test_qkv_rope(M, row_tiles, Hq, Hkv, D, K, fp8, bias):
    g = torch.Generator(device=DEV).manual_seed(M * 7 + K)
    x = torch.randn(M, K + 8, device=DEV, generator=g).bfloat16()[:, :K]  # rows further apart than they are long
    N = (Hq + 2 * Hkv) * D
    w = (torch.randn(N, K, device=DEV, generator=g) / math.sqrt(K)).bfloat16()
    b = torch.randn(N, device=DEV, generator=g).bfloat16() if bias else None
    pos = torch.randint(0, 500, (M + 3,), device=DEV, generator=g, dtype=torch.int32)
    slots = torch.randperm(40 * 32, device=DEV, generator=g)[:M + 3].long()
    if M > 1:
        slots[M - 1] = -1  # a retired row: nothing is written
    tab = ops.RotaryTable(D, 512, 1e4, DEV)
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
    caches = [ops.alloc_kv_cache(40, Hkv, D, dt, DEV) for _ in range(2)]
    q = sk.qkv_rope(x, w, b, pos, slots, tab, *caches[0], Hq, Hkv, D, row_tiles)
    y = x.double() @ w.double().t()
    if bias:
        y = y + b.double()
    want = y.bfloat16().view(M, Hq + 2 * Hkv, D).contiguous()
    ops.rope_and_cache_write_(want, pos[:M], slots[:M], tab, *caches[1], Hq, Hkv)
    # a rotated value holds its partner's rounding too, whatever its own size: one step of values below 8 is 2^-5
    _close(q, want[:, :Hq].double(), bits=5)
    for got, ref in zip(*caches):  # fp8: a value next to a rounding edge of 3 bits of mantissa may take the other one
        _close(got.float(), ref.float().double(), bits=2 if fp8 else 5)
        assert int(((got.float() != 0) != (ref.float() != 0)).sum()) < 3
        if M > 1:
            written = got if got.shape[2] == 32 else got.transpose(2, 3)
            untouched = torch.ones(40 * 32, dtype=torch.bool, device=DEV)
            untouched[slots[:M - 1]] = False
            assert not written.float().transpose(1, 2).reshape(40 * 32, -1)[untouched].any()


@pytest.mark.parametrize("M,row_tiles", [(1, 1), (16, 1), (17, 2), (33, 1), (100, 2)])
@pytest.mark.parametrize("Hq,Hkv,D,K,fp8,bias", [(12, 2, 128, 1536, False, True), (12, 2, 128, 1536, True, True), (8, 1, 256, 2304, True, False),
                                                 (3, 3, 16, 64, False, False), (1, 1, 128, 5120, False, True)])
def test_every_rounding(M, row_tiles, Hq, Hkv, D, K, fp8, bias):
    """Products in sixteenths are exact in fp32, in any order: bit for bit the bf16 projection, lo c - r(hi s) and hi c + r(lo s) rounded to
    bf16, and on an fp8 cache those of them that it holds."""
    g = torch.Generator(device=DEV).manual_seed(M * 7 + K)
    sixteenths = lambda n, *shape: torch.randint(-n, n + 1, shape, device=DEV, generator=g).float() / 16
    x, N = sixteenths(5, M, K).bfloat16(), (Hq + 2 * Hkv) * D
    w, b = sixteenths(2, N, K).bfloat16(), sixteenths(9, N).bfloat16() if bias else None
    pos, slots = torch.randint(0, 500, (M,), device=DEV, generator=g, dtype=torch.int32), torch.randperm(8 * 32, device=DEV, generator=g)[:M].long()
    tab = ops.RotaryTable(D, 512, 1e4, DEV)
    kc, vc = ops.alloc_kv_cache(8, Hkv, D, torch.float8_e4m3fn if fp8 else torch.bfloat16, DEV)
    q = sk.qkv_rope(x, w, b, pos, slots, tab, kc, vc, Hq, Hkv, D, row_tiles)
    y = x.float() @ w.float().t() + (b.float() if bias else 0.0)
    y = y.bfloat16().float().view(M, Hq + 2 * Hkv, 2, D // 2)
    lo, hi, (c, s) = y[:, :Hq + Hkv, 0], y[:, :Hq + Hkv, 1], (t[pos.long()][:, None] for t in (tab.cos, tab.sin))
    rot = torch.cat([lo.double() * c.double() - (hi * s).double(), hi.double() * c.double() + (lo * s).double()], -1).float().bfloat16()
    assert torch.equal(q, rot[:, :Hq])
    v = y[:, Hq + Hkv:].reshape(M, Hkv, D).bfloat16()
    assert torch.equal(kc.float()[slots // 32, :, slots % 32], rot[:, Hq:].to(kc.dtype).float())
    assert torch.equal(vc.float()[slots // 32, :, :, slots % 32], v.to(vc.dtype).float())


def test_rule():
    assert sk.qkv_row_tiles(24, 1536, 2048, 128) == 1 and sk.qkv_row_tiles(32, 1536, 2048, 128) == 1
    assert sk.qkv_row_tiles(33, 1536, 2048, 128) == 2 and sk.qkv_row_tiles(64, 1536, 2048, 128) == 2
    assert sk.qkv_row_tiles(65, 1536, 2048, 128) == 0 and sk.qkv_row_tiles(24, 2048, 2560, 128) == 0
    assert sk.qkv_row_tiles(16, 2304, 4096, 256) == 1 and sk.qkv_row_tiles(9, 3584, 4608, 128) == 0
    assert sk.qkv_row_tiles(9, 1536 + 32, 2048, 128) == 0


@pytest.mark.parametrize("row_tiles", [1, 2])
def test_without_rotation_the_table_is_not_needed(row_tiles):
    """Positions far out and a table of one position of smaller heads: nothing of it is read. Sums are exact, as above."""
    g = torch.Generator(device=DEV).manual_seed(row_tiles)
    sixteenths = lambda n, *shape: torch.randint(-n, n + 1, shape, device=DEV, generator=g).float() / 16
    M, Hq, Hkv, D, K = 19, 3, 2, 128, 256
    x, w, b = sixteenths(5, M, K).bfloat16(), sixteenths(2, (Hq + 2 * Hkv) * D, K).bfloat16(), sixteenths(9, (Hq + 2 * Hkv) * D).bfloat16()
    pos, slots = torch.full((M,), 1 << 30, device=DEV, dtype=torch.int32), torch.arange(M, device=DEV)
    kc, vc = ops.alloc_kv_cache(1, Hkv, D, torch.bfloat16, DEV)
    q = sk.qkv_rope(x, w, b, pos, slots, ops.RotaryTable(16, 1, 1e4, DEV), kc, vc, Hq, Hkv, D, row_tiles, do_rope=False)
    y = (x.float() @ w.float().t() + b.float()).bfloat16().view(M, Hq + 2 * Hkv, D)
    assert torch.equal(q, y[:, :Hq]) and torch.equal(kc[0, :, :M].transpose(0, 1), y[:, Hq:Hq + Hkv])
    assert torch.equal(vc[0, :, :, :M].permute(2, 0, 1), y[:, Hq + Hkv:])
