"""Paged prefill attention in ranges of keys, for few and for many (request, key head) groups: the same as in one range."""
import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.ops import attention as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,hkv,group", [(1, 1, 7), (1, 2, 6), (7, 1, 2), (2, 4, 8), (5, 2, 3), (9, 1, 1)])  # below and from 8 groups on
@pytest.mark.parametrize("splits", [2, 7, 32])
def test_groups(B, hkv, group, splits, monkeypatch):
    g = torch.Generator(device="cuda").manual_seed(B * hkv)
    q_lens = [(37 * (b + 1)) % 300 + 1 for b in range(B)]
    k_lens = [n + 61 * b * b for b, n in enumerate(q_lens)]
    pages = [(k + 31) // 32 for k in k_lens]
    P = sum(pages)
    kc = torch.randn(P, hkv, 32, 128, device="cuda", generator=g).bfloat16()
    vc = torch.randn(P, hkv, 128, 32, device="cuda", generator=g).bfloat16()
    perm = torch.randperm(P, generator=torch.Generator().manual_seed(B)).int()
    bt = torch.zeros(B, max(pages), dtype=torch.int32)
    at = 0
    for b, n in enumerate(pages):
        bt[b, :n] = perm[at:at + n]
        at += n
        if k_lens[b] % 32:  # slots behind the context
            kc[bt[b, n - 1].item(), :, k_lens[b] % 32:] = float("nan")
            vc[bt[b, n - 1].item(), :, :, k_lens[b] % 32:] = float("nan")
    cu = lambda x: torch.tensor([0] + x, device="cuda").cumsum(0).int()
    q = torch.randn(sum(q_lens), hkv * group, 128, device="cuda", generator=g).bfloat16()
    out = []
    for n in (1, splits):
        monkeypatch.setattr(A, "paged_prefill_splits", lambda *a: n)
        out.append(ops.flash_attn_paged_prefill(q, kc, vc, bt.cuda(), cu(q_lens), cu(k_lens), max(q_lens)).double())
    # the same bf16 weights up to a factor, fp32 sums in another order, one rounding to bf16 of values up to 6
    assert float((out[0] - out[1]).abs().max()) < 0.03
    at = 0
    for b, (n, k) in enumerate(zip(q_lens, k_lens)):
        pg = bt[b, :pages[b]].long().cuda()
        kk = kc[pg].double().permute(1, 0, 2, 3).reshape(hkv, -1, 128)[:, :k].repeat_interleave(group, 0)
        vv = vc[pg].double().permute(1, 0, 3, 2).reshape(hkv, -1, 128)[:, :k].repeat_interleave(group, 0)
        s = torch.matmul(q[at:at + n].double().transpose(0, 1), kk.transpose(1, 2).contiguous()) / 128 ** 0.5
        hide = torch.arange(k, device="cuda")[None] > torch.arange(n, device="cuda")[:, None] + k - n
        want = torch.matmul(s.masked_fill(hide, float("-inf")).softmax(-1), vv).transpose(0, 1)
        assert float((out[1][at:at + n] - want).abs().max()) < 0.03
        at += n
