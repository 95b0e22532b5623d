"""The o projection that combines the decode attention's partial results itself: bit for bit the two apart."""
import math

import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.ops import decode_skinny as sk

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Hq,Hkv,D,N", [(12, 2, 128, 1536), (14, 2, 64, 896), (1, 1, 64, 7), (6, 6, 256, 40), (64, 8, 128, 300), (28, 4, 128, 3584)])
@pytest.mark.parametrize("ctx", [[1], [0], [32], [193], [640], [2000], [9000], [24000]])
@pytest.mark.parametrize("fp8", [False, True])
def test_bits_of_the_two_apart(Hq, Hkv, D, N, ctx, fp8):
    g = torch.Generator(device=DEV).manual_seed(sum(ctx) + D)
    M, width = len(ctx), -(-max(max(ctx), 1) // 32) + 1
    bt = (torch.randperm(M * width, device=DEV, generator=g)).view(M, width).int()
    cl = torch.tensor(ctx, dtype=torch.int32, device=DEV)
    caches = []
    for c in ops.alloc_kv_cache(M * width, Hkv, D, torch.bfloat16, DEV):
        c.normal_(generator=g)
        caches.append(ops.attention.to_fp8(c) if fp8 else c)
    q = torch.randn(M, Hq, D, device=DEV, generator=g).bfloat16()
    w = (torch.randn(N, Hq * D, device=DEV, generator=g) / math.sqrt(Hq * D)).bfloat16()
    r = torch.randn(M, N, device=DEV, generator=g).bfloat16()
    items = ops.DecodeItems(M, Hq, Hkv, D, torch.device(DEV), max_context=width * 32).fill_(cl)
    want = sk.linear_residual(ops.paged_attention_decode(q, *caches, bt, cl, items=items).view(M, Hq * D), w, r)
    items.part_o.fill_(float("nan")), items.part_ml.fill_(float("nan"))  # nothing is left over from the call before
    x = torch.full((M, Hq, D), float("nan"), device=DEV).bfloat16()
    ops.paged_attention_decode(q, *caches, bt, cl, items=items, combine=False, out=x)
    got = sk.parts_residual(x, items, w, r)
    assert torch.equal(got, want) and bool(torch.isfinite(got.float()).all())
    assert int(items.arrived.abs().sum()) == 0
    n = items.rows[:, 1].tolist()
    assert all(1 <= k for k in n) and items.rows[:, 0].tolist() == [0] + n[:-1]
