"""Windowed paged prefill against fp64: few and many (request, key head) groups, more tiles of keys than page ids are fetched at once."""
import pytest
import torch

from areal_vllm_amd.ops import window_attention as wattn

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,G,group", [(1, 1, 4), (1, 2, 6), (7, 1, 1), (3, 3, 2)])  # below and from 8 groups on
@pytest.mark.parametrize("window,keep,chunk", [(2500, 0, 0), (2300, 130, 0), (100, 4, 0), (0, 0, 2600), (0, 0, 0)])
@pytest.mark.parametrize("biased", [False, True])
def test_against_fp64(B, G, group, window, keep, chunk, biased):
    g = torch.Generator(device=DEV).manual_seed(B * 100 + window + chunk)
    H = G * group
    q_lens = [(53 * (b + 1)) % 190 + 3 for b in range(B)]
    k_lens = [n + (2900 - 700 * (b % 3)) for b, n in enumerate(q_lens)]  # up to 48 tiles of 64 keys
    pages = [(k + 31) // 32 for k in k_lens]
    P = sum(pages)
    kc = torch.randn(P, G, 32, 128, device=DEV, generator=g).bfloat16()
    vc = torch.randn(P, G, 128, 32, device=DEV, generator=g).bfloat16()
    perm = torch.randperm(P, generator=torch.Generator().manual_seed(B)).int()
    bt, at = torch.zeros(B, max(pages), dtype=torch.int32), 0
    for b, n in enumerate(pages):
        bt[b, :n] = perm[at:at + n]
        at += n
        if k_lens[b] % 32:  # slots behind the context
            kc[bt[b, n - 1].item(), :, k_lens[b] % 32:] = float("nan")
            vc[bt[b, n - 1].item(), :, :, k_lens[b] % 32:] = float("nan")
    cu = lambda x: torch.tensor([0] + x, device=DEV).cumsum(0).int()
    q = torch.randn(sum(q_lens), H, 128, device=DEV, generator=g).bfloat16()
    bias = None
    if biased:
        bias = tuple((torch.rand(H, device=DEV, generator=g) * s).bfloat16() for s in (2.0, 0.1))
    shape = wattn.ScoreShape(scale=128 ** -0.5, window=window, keep_first=keep, chunk=chunk)
    out = wattn.window_attention_standard(q, kc, vc, bt.to(DEV), cu(q_lens), cu(k_lens), torch.tensor(k_lens, device=DEV).int(), max(q_lens),
                                          shape, log_bias=bias).double()
    at = 0
    for b, (n, k) in enumerate(zip(q_lens, k_lens)):
        pg = bt[b, :pages[b]].long().to(DEV)
        kk = kc[pg].double().permute(1, 0, 2, 3).reshape(G, -1, 128)[:, :k].repeat_interleave(group, 0)
        vv = vc[pg].double().permute(1, 0, 3, 2).reshape(G, -1, 128)[:, :k].repeat_interleave(group, 0)
        i, j = torch.arange(k - n, k, device=DEV)[:, None], torch.arange(k, device=DEV)[None]
        s = torch.matmul(q[at:at + n].double().transpose(0, 1), kk.transpose(1, 2).contiguous()) / 128 ** 0.5
        if biased:
            s = s - bias[0].double()[:, None, None] * torch.log1p(bias[1].double()[:, None, None] * (i - j).clamp(min=0))
        lo = torch.zeros_like(i)
        if window:
            lo = (i - window + 1).clamp(min=0)
        if chunk:
            lo = torch.maximum(lo, i // chunk * chunk)
        hide = (j > i) | ((j < lo) & (j >= keep))
        want = torch.matmul(s.masked_fill(hide, float("-inf")).softmax(-1), vv).transpose(0, 1)
        # weights at 16 bits of mantissa, one rounding to bf16 of values up to 6
        assert float((out[at:at + n] - want).abs().max()) < 0.03
        at += n
