"""Rotation and cache write of many tokens at once: the same bits as in pieces that the kernel of one workgroup a token takes."""
import pytest
import torch

from areal_vllm_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,D", [(12, 2, 128), (3, 1, 64), (4, 2, 256), (2, 2, 16)])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("order", ["prompts", "any"])
def test_same_as_in_pieces(hq, hkv, D, fp8, order):
    T = 8192 + 45
    g = torch.Generator().manual_seed(D)
    if order == "prompts":  # lengths around whole eights and pages, the first slot of a prompt anywhere in its page
        pos, slots, page = [], [], 0
        for n in torch.randint(1, 100, (T,), generator=g).tolist():
            n = min(n, T - len(pos))
            first = int(torch.randint(0, 40, (1,), generator=g))
            pos += range(first, first + n)
            slots += [page * 32 + first + i for i in range(n)]
            page += (first + n + 31) // 32
        pos, slots = torch.tensor(pos), torch.tensor(slots)
        pages = page + 1
        perm = torch.randperm(pages, generator=g)
        slots = perm[slots // 32] * 32 + slots % 32
        slots[torch.randint(0, T, (40,), generator=g)] = -1
    else:
        pages = T // 16
        slots, pos = torch.randperm(pages * 32, generator=g)[:T], torch.randint(0, 3000, (T,), generator=g)
    pos, slots = pos.int().cuda(), slots.cuda()
    qkv = torch.randn(T, hq + 2 * hkv, D, generator=g).bfloat16().cuda()
    table = ops.RotaryTable(D, 2000, 1e4, "cuda")  # positions beyond the table take its last row
    out = []
    for step in (T, 4000):
        x = qkv.clone()
        kc, vc = ops.alloc_kv_cache(pages, hkv, D, torch.float8_e4m3fn if fp8 else torch.bfloat16, "cuda")
        kc.view(torch.uint8).fill_(7)
        vc.view(torch.uint8).fill_(7)
        for at in range(0, T, step):
            ops.rope_and_cache_write_(x[at:at + step], pos[at:at + step].contiguous(), slots[at:at + step].contiguous(), table, kc, vc, hq, hkv)
        out.append((x, kc.view(torch.uint8), vc.view(torch.uint8)))
    for a, b in zip(*out):
        assert torch.equal(a, b)
