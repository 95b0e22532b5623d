"""The layers of a short prefill from one native call, against the single launches; the one upload of a prefill plan."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.inference.model_runner import ModelRunner
from areal_vllm_amd.models.config import ModelConfig
from areal_vllm_amd.models.transformer import Transformer


@pytest.mark.gpu
@pytest.mark.parametrize("family,extra", [("qwen2", dict(qkv_bias=True)), ("qwen3", dict(qk_norm=True)),
                                          ("gemma", dict(gemma_norm=True, hidden_act="gelu_tanh"))])
@pytest.mark.parametrize("layers,new,prefix,fp8", [(1, [1], [40], False), (2, [93, 5, 40], [200, 0, 33], False), (3, [160, 161], [64, 7], True)])
def test_same_bits_as_the_single_launches(family, extra, layers, new, prefix, fp8, monkeypatch):
    torch.manual_seed(1)
    cfg = ModelConfig(family=family, vocab_size=512, hidden_size=256, n_layers=layers, n_q_heads=4, n_kv_heads=2, head_dim=128,
                      intermediate_size=448, max_position_embeddings=2048, **extra)
    m = Transformer(cfg, dtype=torch.bfloat16, device=torch.device("cuda"))
    m.requires_grad_(False)
    m.flatten()
    for n, p in m.named_parameters():
        p.copy_(torch.randn_like(p) * (0.05 if p.dim() > 1 else 0.1) + (p.dim() == 1 and "bias" not in n))
    rows = len(new)
    ctx = np.add(prefix, new)
    need = [-(-int(c) // 32) for c in ctx]
    bt = np.zeros((rows, max(need)), np.int32)
    at = 0
    for b, k in enumerate(need):
        bt[b, :k] = np.arange(at, at + k)
        at += k
    pos = np.concatenate([np.arange(c, c + n) for c, n in zip(prefix, new)]).astype(np.int32)
    row = np.repeat(np.arange(rows), new)
    cu = lambda x: np.concatenate([[0], np.cumsum(x)]).astype(np.int32)
    plan = dict(input_ids=np.random.RandomState(0).randint(0, 512, sum(new)).astype(np.int32), positions=pos,
                slot_mapping=bt[row, pos // 32].astype(np.int64) * 32 + pos % 32, cu_q=cu(new), cu_k=cu(ctx), max_q=max(new),
                has_prefix=True, block_tables=bt, req_ids=np.arange(rows), temperature=np.zeros(rows, np.float32),
                top_p=np.ones(rows, np.float32), top_k=np.full(rows, 1 << 30), sample=np.ones(rows, np.int32),
                logit_rows=cu(new)[1:].astype(np.int64) - 1)
    native, calls, out = ops.prefill_layers.run, [], []

    def counted(*a):
        r = native(*a)
        calls.append(r is not None)
        return r

    for run in (counted, lambda *a: None):
        monkeypatch.setattr(ops.prefill_layers, "run", run)
        r = ModelRunner(m, num_pages=64, max_context=1024, max_batch=4, kv_dtype=torch.float8_e4m3fn if fp8 else torch.bfloat16)
        g = torch.Generator(device="cuda").manual_seed(1)
        for pair in r.kv:
            for t in pair:
                x = torch.randn(t.shape, device="cuda", generator=g).bfloat16() * 0.3
                t.copy_(ops.attention.to_fp8(x) if fp8 else x)
        tok, lp = r.prefill(plan)
        out.append([torch.from_numpy(tok), torch.from_numpy(lp), r.kept_logits.clone()] + [t.view(torch.uint8).clone() for kv in r.kv for t in kv])
    assert calls == [True]
    for a, b in zip(*out):
        assert torch.equal(a, b)


def test_upload():
    arrays = dict(a=np.arange(5, dtype=np.int32), b=np.ones((3, 2), np.float32), c=np.arange(12).reshape(3, 4)[:, ::2],
                  d=np.zeros(0, np.int64), e=np.arange(7, dtype=np.int64), f=np.array([True, False, True]))
    got = ModelRunner._upload(SimpleNamespace(device=torch.device("cpu")), arrays)
    for k, v in arrays.items():
        assert got[k].numpy().dtype == v.dtype and np.array_equal(got[k].numpy(), v) and got[k].shape == v.shape


@pytest.mark.gpu
@pytest.mark.parametrize("layers,odd", [(1, None), (2, None), (3, None), (8, None), (9, None), (13, None), (3, 0), (3, 1), (9, 2), (9, 8)])
def test_layers_in_several_calls(layers, odd, monkeypatch):
    """Every number of layers around those of the first calls, and a layer whose weight is off the 16-byte grid in each of them, for which
    the single launches take over from the start: their bits, and near the numbers of the layers' other path."""
    torch.manual_seed(1)
    cfg = ModelConfig(family="qwen2", vocab_size=512, hidden_size=128, n_layers=layers, n_q_heads=2, n_kv_heads=1, head_dim=128,
                      intermediate_size=192, max_position_embeddings=512, qkv_bias=True)
    m = Transformer(cfg, dtype=torch.bfloat16, device=torch.device("cuda"))
    m.requires_grad_(False)
    m.flatten()
    for n, p in m.named_parameters():
        p.copy_(torch.randn_like(p) * (0.05 if p.dim() > 1 else 0.1) + (p.dim() == 1 and "bias" not in n))
    plan = dict(input_ids=np.arange(5, dtype=np.int32), positions=np.arange(40, 45, dtype=np.int32), slot_mapping=np.arange(40, 45),
                cu_q=np.array([0, 5], np.int32), cu_k=np.array([0, 45], np.int32), max_q=5, has_prefix=True,
                block_tables=np.arange(2, dtype=np.int32)[None], req_ids=np.arange(1), temperature=np.zeros(1, np.float32),
                top_p=np.ones(1, np.float32), top_k=np.full(1, 1 << 30), sample=np.ones(1, np.int32), logit_rows=np.arange(5))
    native, calls, out = ops.prefill_layers.run, [], []

    def counted(*a):
        r = native(*a)
        calls.append(r is not None)
        return r

    if odd is not None:
        w = m.layers[odd].mlp.down if odd % 2 else m.layers[odd].ln2
        moved = torch.empty(w.numel() + 4, dtype=w.dtype, device="cuda")[4:].view_as(w)  # 8 bytes past the grid
        w.data = moved.copy_(w)
    for run, fused in ((counted, True), (lambda *a: None, True), (None, False)):
        monkeypatch.setattr(ops.prefill_layers, "run", run)
        r = ModelRunner(m, num_pages=2, max_context=64, max_batch=1)
        if not fused:
            r._prefill_fused = lambda rows: False
        for pair in r.kv:
            for t in pair:
                t.copy_(torch.linspace(-1, 1, t.numel(), device="cuda").view_as(t))
        r.prefill(plan)
        out.append((r.kept_logits.clone(), [t.clone() for kv in r.kv for t in kv]))
    assert calls == [odd is None]
    (la, ca), (ls, cs), (lb, cb) = out
    assert torch.equal(la, ls) and all(torch.equal(a, b) for a, b in zip(ca, cs))
    # 16-bit roundings of the layers' products (library against split sums) add up over the layers: some steps of 2^-8
    assert float((la - lb).norm() / lb.norm()) < 2.0 ** -8 * (2 + layers)
    for a, b in zip(ca, cb):
        assert float((a.float() - b.float()).norm() / b.float().norm()) < 2.0 ** -8 * (2 + layers)
