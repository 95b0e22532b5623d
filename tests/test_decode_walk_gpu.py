"""Decode attention on work items: waves that walk more pages than they hold ids of, and every value of an fp8 cache."""
import math

import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.ops import attention as A

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,fp8", [(64, False), (128, True)])
def test_items_of_more_than_512_pages(D, fp8):
    """600 rows and one key head: an item is a whole row, so a wave walks 65 to 68 pages and fetches ids a second time. The
    rows share 600 pages, each in an order of its own."""
    g = torch.Generator().manual_seed(1)
    B, Hq = 600, 5
    ctx = torch.randint(513 * 32, 540 * 32, (B,), generator=g, dtype=torch.int32)
    ctx[:3] = torch.tensor([512 * 32, 512 * 32 + 1, 513 * 32])
    bt = torch.stack([torch.randperm(600, generator=g)[:541] + 1 for _ in range(B)]).int()
    kc, vc = ops.alloc_kv_cache(601, 1, D, torch.bfloat16, "cpu")
    kc.copy_(torch.randn(kc.shape, generator=g))
    vc.copy_(torch.randn(vc.shape, generator=g))
    if fp8:
        kc, vc = kc.to(A.FP8), vc.to(A.FP8)
    q = (2 * torch.randn(B, Hq, D, generator=g)).bfloat16()
    d = [t.to(DEV) for t in (q, kc, vc, bt, ctx)]
    items = ops.DecodeItems(B, Hq, 1, D, torch.device(DEV)).fill_(d[4])
    assert int((items.items[:, 2] - items.items[:, 1]).max()) > 512
    out = ops.paged_attention_decode(*d, items=items).float().cpu()
    some = [0, 1, 2, 150, 599]
    ref = A.paged_decode_ref(q[some], kc, vc, bt[some], ctx[some], 1 / math.sqrt(D)).float()
    # P in bf16 (2^-9 relative per weight) and a bf16 result: errors of a few 2^-9 of values of order one
    assert (out[some] - ref).abs().max() < 2e-2


def test_every_fp8_value_is_read_exactly():
    kc, vc = ops.alloc_kv_cache(9, 1, 64, A.FP8, DEV)
    every = torch.arange(256, dtype=torch.uint8, device=DEV)
    for c in (kc, vc):
        c.view(torch.uint8).view(-1, 256).copy_(every)
    slots = torch.arange(9 * 32, device=DEV)
    k, v = ops.cache_gather(kc, vc, slots)
    want_k = kc.view(9 * 32, 64).to(torch.bfloat16)  # pages [32][64]
    want_v = vc.view(9, 64, 32).to(torch.bfloat16).transpose(1, 2).reshape(9 * 32, 64)
    for got, want in ((k[:, 0], want_k), (v[:, 0], want_v)):
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(0.5), want.nan_to_num(0.5))
