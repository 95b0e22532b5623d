"""Flash attention forward and backward at the edges of their tiles, with the dK / dV work of a key block shared by several
workgroups, under scales of either sign and rows that see no key."""
import math

import numpy as np
import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.ops import attention as A

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


def _ref(q, k, v, lq, lk, scale, causal):
    """fp64 attention [Tq, Hq, D]; rows without a key give zero."""
    g, outs, a, b = q.shape[1] // k.shape[1], [], 0, 0
    for m, n in zip(lq, lk):
        qq, kk, vv = (x.transpose(0, 1) for x in (q[a:a + m], k[b:b + n].repeat_interleave(g, 1), v[b:b + n].repeat_interleave(g, 1)))
        s = torch.matmul(qq, kk.transpose(1, 2)) * scale
        if causal:
            i, j = torch.arange(m, device=q.device)[:, None], torch.arange(n, device=q.device)[None, :]
            s = s.masked_fill(j > i + n - m, -math.inf)
        p = torch.nan_to_num(torch.softmax(s, -1), nan=0.0)
        outs.append(torch.matmul(p, vv).transpose(0, 1))
        a, b = a + m, b + n
    return torch.cat(outs)


@pytest.mark.parametrize("Hq,Hkv", [(6, 1), (14, 2), (3, 3)])
@pytest.mark.parametrize("lq,lk", [([1], [1]), ([31, 32, 33], None), ([127, 128, 129], None), ([64, 63, 65, 300], None),
                                   ([5, 130], [700, 131]), ([200, 1, 0], [40, 64, 3]), ([1500], None)])
@pytest.mark.parametrize("scale,causal", [(None, True), (None, False), (-0.11, True)])
def test_forward_and_gradients(Hq, Hkv, lq, lk, scale, causal):
    lk = lk or lq
    g = torch.Generator(device=DEV).manual_seed(sum(lq) + Hq)
    q, k, v = (torch.randn(sum(l), h, 128, device=DEV, generator=g).bfloat16().requires_grad_() for l, h in
               ((lq, Hq), (lk, Hkv), (lk, Hkv)))
    cu = [torch.tensor([0] + np.cumsum(l).tolist(), dtype=torch.int32, device=DEV) for l in (lq, lk)]
    assert A.flash_bwd_parts(sum(lk), max(lk), Hq, Hkv) == Hq // Hkv  # every query head a workgroup of its own
    out = ops.flash_attn_varlen_sep(q, k, v, *cu, max(lq), max(lk), scale, causal)
    d = torch.randn(out.shape, device=DEV, generator=g).bfloat16()
    grads = torch.autograd.grad(out, (q, k, v), d, retain_graph=True)
    again = torch.autograd.grad(out, (q, k, v), d)
    assert all(torch.equal(x, y) for x, y in zip(grads, again))  # no sum depends on the order of arrival
    r = [x.detach().double().requires_grad_() for x in (q, k, v)]
    want = _ref(*r, lq, lk, scale or 128 ** -0.5, causal)
    refs = torch.autograd.grad(want, r, d.double())
    out, want = out.detach(), want.detach()
    # P, dS, O and the gradients pass through bf16 once (2^-9 each, relative to a row's largest value)
    for x, y in zip((out, *grads), (want, *refs)):
        assert float((x.double() - y).abs().max()) <= 2e-2 * max(1.0, float(y.abs().max())), (x.shape, float(y.abs().max()))
        # (a row with one key: dP - delta is the difference of two fp32 sums below 64 in size, 1e-5, where zero is exact)
        assert float((x.double() - y).norm()) <= 8e-3 * float(y.norm()) + 1e-5 * x.numel() ** 0.5


def test_parts_cover_the_heads():
    for g in range(1, 17):
        for tk in (1, 700, 5000, 24576, 200000):
            for mk in (min(tk, 1000), tk):
                p = A.flash_bwd_parts(tk, mk, 2 * g, 2)
                assert 1 <= p <= g


def test_scores_that_keep_growing_are_rescaled():
    """Keys whose scores grow from tile to tile, by a little and by much: every tile rescales what came before it."""
    T = 1024
    q = torch.ones(T, 2, 128, device=DEV).bfloat16()
    k = (torch.arange(T, device=DEV)[:, None, None] * 2e-3 * torch.ones(T, 1, 128, device=DEV)).bfloat16()
    v = torch.randn(T, 1, 128, device=DEV).bfloat16()
    cu = torch.tensor([0, T], dtype=torch.int32, device=DEV)
    for scale in (0.02, 1.0, 0.0):
        out, lse = ops.flash_attn_varlen(q, k, v, cu, cu, T, scale=scale)
        ref, ref_lse = A.attention_varlen_ref(q.double(), k.double(), v.double(), cu, cu, scale)
        assert float((out.float() - ref).abs().max()) < 2e-2
        assert float((lse - ref_lse).abs().max()) < 2e-3 * max(1.0, float(ref_lse.abs().max()))


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("T,row", [(64, 40), (130, 3), (700, 333), (1200, 1199)])
def test_a_row_depends_on_its_own_query_only(T, row, causal):
    """Bit for bit the same output and log-sum-exp whatever the other queries of its tile are."""
    g = torch.Generator(device=DEV).manual_seed(T)
    q, k, v = (torch.randn(T, h, 128, device=DEV, generator=g).bfloat16() for h in (4, 2, 2))
    cu = torch.tensor([0, T], dtype=torch.int32, device=DEV)
    got = []
    for size in (0.0, 1.0, 12.0):  # neighbours whose maxima stand still, drift, and jump from tile to tile
        other = (torch.randn(T, 4, 128, device=DEV, generator=g) * size).bfloat16()
        other[row] = q[row]
        out, lse = ops.flash_attn_varlen(other, k, v, cu, cu, T, causal=causal)
        got.append((out[row], lse[:, row]))
    for out, lse in got[1:]:
        assert torch.equal(out, got[0][0]) and torch.equal(lse, got[0][1])


@pytest.mark.parametrize("D", [128, 256])
@pytest.mark.parametrize("n", [300, 3000])
def test_rows_of_no_sequence_get_zero_gradients(D, n):
    g = torch.Generator(device=DEV).manual_seed(n)
    lead, tail, Hq, Hkv = 5, 140, 4, 2
    T = lead + n + tail
    qkv = torch.randn(T, Hq + 2 * Hkv, D, device=DEV, generator=g).bfloat16()
    d = torch.randn(T, Hq, D, device=DEV, generator=g).bfloat16()
    cu = torch.tensor([lead, lead + n // 3, lead + n], dtype=torch.int32, device=DEV)
    none = torch.ones(T, dtype=torch.bool, device=DEV)
    none[lead:lead + n] = False

    def fresh():  # what is allocated next holds NaN
        for shape in ((T, Hq + 2 * Hkv, D), (T, Hq, D), (T, Hkv, D), (T, Hkv, D)):
            torch.full(shape, math.nan, dtype=torch.bfloat16, device=DEV)

    grads = []
    for x in (qkv, qkv[lead:lead + n]):  # with the rows of no sequence, and without them
        x = x.clone().requires_grad_()
        o = 0 if x.shape[0] == T else lead
        y = ops.flash_attn_varlen_qkv(x, cu - o, n, Hq, Hkv)
        fresh()
        grads.append(torch.autograd.grad(y, x, d[o:o + y.shape[0]])[0])
    assert bool((grads[0][none] == 0).all()) and torch.equal(grads[0][~none], grads[1])

    q, k, v = (t.contiguous().requires_grad_() for t in qkv.split([Hq, Hkv, Hkv], 1))
    more = torch.cat([k.detach(), k.detach()]).requires_grad_()  # more keys than queries, the second half of no sequence
    y = ops.flash_attn_varlen_sep(q, more, torch.cat([v, v]), cu, cu, n, n)
    fresh()
    dq, dk = torch.autograd.grad(y, (q, more), d)
    assert bool((dq[none] == 0).all()) and bool((dk[:T][none] == 0).all()) and bool((dk[T:] == 0).all())
    assert torch.equal(dq[~none], grads[1][:, :Hq]) and torch.equal(dk[:T][~none], grads[1][:, Hq:Hq + Hkv])
