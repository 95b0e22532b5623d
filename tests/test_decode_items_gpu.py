"""Decode attention on work items: the items cover every row's pages once, and the walk equals attention in fp32."""
import math

import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.ops import attention as A

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


def _setup(ctx, Hq, Hkv, D, fp8, seed):
    g = torch.Generator().manual_seed(seed)
    need = [(c + 31) // 32 for c in ctx]
    width = max(need + [1]) + 1
    bt = torch.zeros(len(ctx), width, dtype=torch.int32)
    perm, at = torch.randperm(sum(need), generator=g) + 1, 0
    for b, n in enumerate(need):
        bt[b, :n] = perm[at:at + n].int()
        at += n
    kc, vc = ops.alloc_kv_cache(sum(need) + 1, Hkv, D, torch.bfloat16, "cpu")
    kc.copy_(torch.randn(kc.shape, generator=g))
    vc.copy_(torch.randn(vc.shape, generator=g))
    if fp8:
        kc, vc = kc.to(A.FP8), vc.to(A.FP8)
    q = torch.randn(len(ctx), Hq + 1, D, generator=g).bfloat16()
    return q, kc, vc, bt, torch.tensor(ctx, dtype=torch.int32)


@pytest.mark.parametrize("Hq,Hkv,D,fp8", [(12, 2, 128, False), (12, 2, 128, True), (32, 4, 128, False), (7, 7, 64, False),
                                          (16, 2, 64, True), (8, 1, 256, False), (16, 1, 256, True)])
@pytest.mark.parametrize("ctx", [[1], [640], list(range(3000, 9000, 100)), [0, 1, 31, 32, 33, 127, 128, 129, 4099], [3000] * 3 + [1] * 1100])
def test_decode_attention_on_items(Hq, Hkv, D, fp8, ctx):
    if len(ctx) > 100 and Hkv == 7:
        pytest.skip("one wide batch a head count is enough")
    q, kc, vc, bt, cl = _setup(ctx, Hq, Hkv, D, fp8, 3)
    d = [t.to(DEV) for t in (q, kc, vc, bt, cl)]
    items = ops.DecodeItems(len(ctx), Hq, Hkv, D, torch.device(DEV)).fill_(d[4])
    tight = ops.DecodeItems(len(ctx), Hq, Hkv, D, torch.device(DEV), max_context=max(ctx)).fill_(d[4])
    assert tight.n_items <= items.n_items and int((tight.items[:, 4] > 0).sum()) == int((items.items[:, 4] > 0).sum())
    # rows' pages: contiguous ranges, in order, of at most one multiple of four pages each
    rows = {}
    parts = set()
    for b, lo, hi, base, n, part in items.items[:, :6].tolist():
        if n:
            rows.setdefault(b, []).append((part - base, lo, hi, n))
            parts.add(part)
    assert sorted(rows) == list(range(len(ctx))) and len(parts) == sum(len(r) for r in rows.values())
    for b, c in enumerate(ctx):
        r = sorted(rows[b])
        assert [x[0] for x in r] == list(range(len(r))) and all(x[3] == len(r) for x in r)
        edges = [0] + [x[2] for x in r]
        assert [x[1] for x in r] == edges[:-1] and edges[-1] == (c + 31) // 32 and all(e % 4 == 0 for e in edges[:-1])
    ref = A.paged_decode_ref(q[:, :Hq], kc, vc, bt, cl, 1 / math.sqrt(D)).float()
    outs = [ops.paged_attention_decode(d[0][:, :Hq], *d[1:], q_row_stride=(Hq + 1) * D, items=items).float().cpu()
            for _ in range(3)]
    # P in bf16 (2^-9 relative per weight) and a bf16 result: errors of a few 2^-9 of values of order one
    assert (outs[0] - ref).abs().max() < 2e-2
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])  # counters are back at zero, order is fixed
    assert int(items.arrived.abs().sum()) == 0
    # the form with a bounded context, as a runner allocates it: its own layout is the same, and so is every bit
    got = ops.paged_attention_decode(d[0][:, :Hq], *d[1:], q_row_stride=(Hq + 1) * D, items=tight).float().cpu()
    assert torch.equal(got, outs[0])


@pytest.mark.parametrize("Hq,Hkv,head_dim,kv,rows,on_items", [
    (4, 1, 64, None, 4, True), (16, 1, 64, None, 4, True), (8, 1, 128, None, 4, True), (16, 1, 128, None, 4, False),
    (16, 1, 128, None, 17, True), (18, 2, 128, A.FP8, 8, False), (18, 2, 128, None, 9, True), (4, 1, 256, None, 4, True),
    (8, 1, 256, None, 4, False), (8, 1, 256, A.FP8, 20, False)])
def test_runner_chooses_items_by_values_a_key_head(Hq, Hkv, head_dim, kv, rows, on_items):
    """Items, or key ranges of one count for all rows where a row has many values to combine; both equal attention in fp32."""
    from areal_vllm_amd.inference.model_runner import ModelRunner
    from areal_vllm_amd.models.config import ModelConfig
    from areal_vllm_amd.models.transformer import Transformer

    cfg = ModelConfig(family="llama", vocab_size=256, hidden_size=256, n_layers=1, n_q_heads=Hq, n_kv_heads=Hkv,
                      head_dim=head_dim, intermediate_size=256, max_position_embeddings=4096)
    model = Transformer(cfg, dtype=torch.bfloat16, device=torch.device(DEV))
    model.requires_grad_(False)
    model.flatten()
    ctx = [(1, 33, 700, 2000)[i % 4] for i in range(rows)]
    q, kc, vc, bt, cl = _setup(ctx, Hq, Hkv, head_dim, kv is not None, 5)
    r = ModelRunner(model, kc.shape[0], 2048, rows, buckets=[rows], kv_dtype=kv)
    st = r._alloc_static(rows)
    assert (st["items"] is not None) == on_items and (st["ws"] is None) == on_items
    d = [t.to(DEV) for t in (q[:, :Hq].contiguous(), kc, vc, bt, cl)]
    if st["items"] is not None:
        st["items"].fill_(d[4])
    got = ops.paged_attention_decode(*d, nsplit=st["nsplit"], workspace=st["ws"], items=st["items"]).float().cpu()
    ref = A.paged_decode_ref(q[:, :Hq], kc, vc, bt, cl, 1 / math.sqrt(head_dim)).float()
    assert (got - ref).abs().max() < 2e-2


@pytest.mark.parametrize("rows,group,common", [(1, 1, 0), (2, 2, 40), (7, 3, 33), (320, 16, 20), (1024, 1024, 8), (1025, 5, 8)])
@pytest.mark.parametrize("D,fp8", [(128, False), (128, True), (64, False), (64, True), (256, False), (256, True)])
def test_pages_that_no_other_row_reads_go_past_the_caches(rows, group, common, D, fp8):
    """Which items are marked: none of those that lie in pages common to a group, all of those behind them (and all results the same)."""
    g = torch.Generator().manual_seed(rows + D)
    ctx = [int(x) for x in torch.randint(32 * common + 1, 32 * common + 700, (rows,), generator=g)]
    q, kc, vc, bt, cl = _setup(ctx, 4, 1, D, fp8, 4)
    order = torch.randperm(rows, generator=g)  # rows of a group are not neighbours
    for i in range(rows):
        bt[order[i], :common] = bt[order[i // group * group], :common]
    d = [t.to(DEV) for t in (q, kc, vc, bt, cl)]
    plain = ops.DecodeItems(rows, 4, 1, D, torch.device(DEV)).fill_(d[4])
    marked = ops.DecodeItems(rows, 4, 1, D, torch.device(DEV)).fill_(d[4], d[3])
    size = {int(r): min(group, rows - i // group * group) for i, r in enumerate(order)}  # rows of its group
    table = {(b, lo): (hi, stream) for b, lo, hi, _, n, _, stream, _ in marked.items.tolist() if n}
    assert len(table) == int((plain.items[:, 4] > 0).sum())
    for (b, lo), (hi, stream) in table.items():
        alone = rows == 1 or (rows <= 1024 and (size[b] == 1 or (lo + hi) // 2 >= common))
        assert stream == int(alone), (b, lo, hi, stream)
    outs = [ops.paged_attention_decode(d[0][:, :4], *d[1:], q_row_stride=5 * D, items=i) for i in (plain, marked)]
    assert torch.equal(*outs)
    ref = A.paged_decode_ref(q[:, :4], kc, vc, bt, cl, 1 / math.sqrt(D)).float()
    assert (outs[0].float().cpu() - ref).abs().max() < 2e-2  # as above


@pytest.mark.parametrize("rows,system,own,per", [(3, 5, 9, 2), (24, 4, 16, 4), (320, 2, 20, 16), (1024, 1, 6, 8), (64, 70, 40, 8)])
@pytest.mark.parametrize("extra", [0, 300])
def test_pages_of_a_prompt_behind_a_common_one(rows, system, own, per, extra):
    """All rows share a system prompt of `system` pages, `per` of them a question of `own` pages behind it: what the rows of one question
    read is theirs in common whichever row of another question came first. Idle rows with one page, all the same, are at the end."""
    g = torch.Generator().manual_seed(rows)
    ctx = [int(x) for x in torch.randint(32 * (system + own) + 1, 32 * (system + own) + 700, (rows,), generator=g)] + [1] * min(extra, 1024 - rows)
    n = len(ctx)
    q, kc, vc, bt, cl = _setup(ctx, 4, 1, 128, False, 4)
    bt[rows:, 0] = 0
    order = torch.randperm(rows, generator=g)
    for i in range(rows):
        bt[order[i], :system] = bt[order[0], :system]
        bt[order[i], system:system + own] = bt[order[i // per * per], system:system + own]
    d = [t.to(DEV) for t in (q, kc, vc, bt, cl)]
    plain = ops.DecodeItems(n, 4, 1, 128, torch.device(DEV)).fill_(d[4])
    marked = ops.DecodeItems(n, 4, 1, 128, torch.device(DEV)).fill_(d[4], d[3])
    pages = [set(bt[b, :(c + 31) // 32].tolist()) for b, c in enumerate(ctx[:rows])]
    readers = {}
    for p in pages:
        for x in p:
            readers[x] = readers.get(x, 0) + 1
    got = [(b, (lo + hi) // 2, stream) for b, lo, hi, _, k, _, stream, _ in marked.items.tolist() if k]
    assert len(got) == int((plain.items[:, 4] > 0).sum())
    for b, mid, stream in got:
        assert stream == int(b >= rows or readers[int(bt[b, mid])] == 1), (b, mid, stream)
    outs = [ops.paged_attention_decode(d[0][:, :4], *d[1:], q_row_stride=5 * 128, items=i) for i in (plain, marked)]
    assert torch.equal(*outs)
