"""Prefills of few tokens: attention over the pages with the keys split over workgroups, the layers on the decode step's
GEMMs, the scoring head."""
import numpy as np
import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.ops import attention as A

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


def _paged(q_lens, k_lens, hkv, fp8, g):
    pages = [(k + 31) // 32 for k in k_lens]
    perm = torch.randperm(sum(pages) + 3, generator=g)[: sum(pages)].to(torch.int32)
    bt = torch.zeros(len(k_lens), max(pages) + 2, dtype=torch.int32)
    at = 0
    for b, n in enumerate(pages):
        bt[b, :n] = perm[at:at + n]
        at += n
    kc = torch.randn(sum(pages) + 3, hkv, 32, 128, generator=g).bfloat16()
    vc = torch.randn(sum(pages) + 3, hkv, 128, 32, generator=g).bfloat16()
    for b, n in enumerate(k_lens):  # slots behind a context hold what must not be read
        if n % 32:
            vc[bt[b, n // 32], :, :, n % 32:] = float("nan")
    if fp8:
        kc, vc = A.to_fp8(kc), A.to_fp8(vc)
    cu = lambda x: torch.tensor(np.concatenate([[0], np.cumsum(x)]), dtype=torch.int32, device=DEV)
    return kc.to(DEV), vc.to(DEV), bt.to(DEV), cu(q_lens), cu(k_lens)


@pytest.mark.parametrize("q_lens,k_lens", [([1], [1]), ([1], [900]), ([93], [904]), ([128], [128]), ([129], [1000]),
                                           ([5, 64, 130], [5, 700, 131]), ([200, 3], [4000, 33])])
@pytest.mark.parametrize("hq,hkv", [(2, 1), (12, 2)])
@pytest.mark.parametrize("fp8", [False, True])
def test_split_keys(q_lens, k_lens, hq, hkv, fp8, monkeypatch):
    g = torch.Generator().manual_seed(sum(k_lens))
    kc, vc, bt, cu_q, cu_k = _paged(q_lens, k_lens, hkv, fp8, g)
    T = sum(q_lens)
    q = torch.randn(T, hq + 2, 128, generator=g).bfloat16().to(DEV)[:, :hq]
    got = {}
    for target in (1, 256, 100000):  # one workgroup a tile, the rule's choice, as many as the page tables allow
        monkeypatch.setattr(A, "PAGED_PREFILL_WORKGROUPS", target)
        monkeypatch.setattr(A, "PAGED_PREFILL_KEYS", 32 if target == 100000 else 128)
        got[target] = ops.flash_attn_paged_prefill(q, kc, vc, bt, cu_q, cu_k, max(q_lens))
    f = lambda t: (t.to(torch.float32) if fp8 else t).double()
    at = 0
    for b, (n, k) in enumerate(zip(q_lens, k_lens)):
        pg = bt[b, : (k + 31) // 32].long()
        kk = f(kc)[pg].permute(1, 0, 2, 3).reshape(hkv, -1, 128)[:, :k].repeat_interleave(hq // hkv, 0)
        vv = f(vc)[pg].permute(1, 0, 3, 2).reshape(hkv, -1, 128)[:, :k].repeat_interleave(hq // hkv, 0)
        s = torch.matmul(q[at:at + n].double().transpose(0, 1), kk.transpose(1, 2)) / 128 ** 0.5
        mask = torch.arange(k, device=DEV)[None] > torch.arange(n, device=DEV)[:, None] + k - n
        want = torch.matmul(s.masked_fill(mask, float("-inf")).softmax(-1), vv).transpose(0, 1)
        for x in got.values():
            # weights in bf16 (2^-9 each, errors of either sign) and an output of size up to max |v| < 6 rounded to bf16
            assert float((x[at:at + n].double() - want).abs().max()) < 0.03
        at += n


@pytest.mark.parametrize("q_lens,k_lens", [([1], [1]), ([128], [128]), ([5, 64, 130], [5, 64, 131]), ([200, 3], [400, 33])])
@pytest.mark.parametrize("splits", [2, 3, 5, 32])
def test_ranges_without_keys(q_lens, k_lens, splits, monkeypatch):
    """More ranges than some request has key tiles, whatever the rule would choose: the same as one range."""
    g = torch.Generator().manual_seed(sum(k_lens))
    kc, vc, bt, cu_q, cu_k = _paged(q_lens, k_lens, 2, False, g)
    q = torch.randn(sum(q_lens), 12, 128, generator=g).bfloat16().to(DEV)
    out = []
    for n in (1, splits):
        monkeypatch.setattr(A, "paged_prefill_splits", lambda *a: n)
        out.append(ops.flash_attn_paged_prefill(q, kc, vc, bt, cu_q, cu_k, max(q_lens)).double())
    # the same bf16 weights up to a factor, fp32 sums in another order, one rounding to bf16 of values up to 6
    assert float((out[0] - out[1]).abs().max()) < 0.03


def test_ranges_only_where_the_walk_is_long():
    f = A.paged_prefill_splits
    assert f(1, 12, 93, 928) > 1 and f(1, 12, 512, 8512) > 1 and f(1, 2, 1, 928) > 1
    assert f(1, 32, 512, 512) == 1 and f(2, 32, 256, 256) == 1 and f(5, 12, 256, 320) == 1 and f(1, 12, 1, 32) == 1


@pytest.mark.parametrize("model", ["dense", "qk_norm", "experts"])
@pytest.mark.parametrize("new,prefix,kv", [([1], [0], None), ([1], [37], None), ([93], [200], None), ([40, 7, 130], [0, 64, 9], None),
                                           ([512], [0], None), ([93], [200], "fp8"), ([50], [0], "fp8")])
def test_layers(model, new, prefix, kv):
    _both_paths(model, new, prefix, kv)


# heads that attention pads to 128 or 256 and hands back as a slice, heads of 256, and rows and norms that the decode step's
# row kernels do not take
@pytest.mark.parametrize("model,heads,fused", [
    ("dense", dict(n_q_heads=14, n_kv_heads=2, head_dim=64), True), ("qk_norm", dict(n_q_heads=4, n_kv_heads=2, head_dim=64), True),
    ("dense", dict(n_q_heads=2, n_kv_heads=1, head_dim=96), True), ("dense", dict(n_q_heads=2, n_kv_heads=1, head_dim=256), True),
    ("qk_norm", dict(n_q_heads=2, n_kv_heads=1, head_dim=96), False),
    ("dense", dict(n_q_heads=120, n_kv_heads=8, head_dim=128), False)])
@pytest.mark.parametrize("new,prefix,kv", [([93], [200], None), ([40, 7, 130], [0, 64, 9], None), ([50, 3], [0, 0], None),
                                           ([93], [200], "fp8")])
def test_layers_of_other_heads(model, heads, fused, new, prefix, kv):
    _both_paths(model, new, prefix, kv, fused, **heads)


def _both_paths(model, new, prefix, kv, fused=True, **heads):
    from areal_vllm_amd.inference.model_runner import ModelRunner
    from areal_vllm_amd.models.config import ModelConfig
    from areal_vllm_amd.models.transformer import Transformer

    torch.manual_seed(0)
    base = dict(vocab_size=512, hidden_size=256, n_layers=3, n_q_heads=4, n_kv_heads=2, head_dim=128, intermediate_size=512,
                max_position_embeddings=2048)
    extra = {"dense": dict(family="qwen2", qkv_bias=True),
             "qk_norm": dict(family="qwen3", qk_norm=True),
             "experts": dict(family="qwen3_moe", qk_norm=True, n_experts=8, n_experts_per_tok=2, moe_intermediate_size=128)}
    cfg = ModelConfig(**{**base, **heads}, **extra[model])
    m = Transformer(cfg, dtype=torch.bfloat16, device=torch.device(DEV))
    m.requires_grad_(False)
    m.eval()
    m.flatten()
    with torch.no_grad():
        for n, p in m.named_parameters():
            p.copy_(torch.randn_like(p) * (0.05 if p.dim() > 1 else 0.1) + (p.dim() == 1 and "bias" not in n))
    rows = len(new)
    out = []
    for limit in (0, 512):
        r = ModelRunner(m, num_pages=64, max_context=1024, max_batch=4,
                        kv_dtype=torch.float8_e4m3fn if kv else torch.bfloat16)
        r.PREFILL_FUSED_MAX_ROWS = limit
        assert r._prefill_fused(sum(new)) == (limit > 0 and fused)
        g = torch.Generator(device=DEV).manual_seed(1)
        for pair in r.kv:
            for t in pair:
                x = torch.randn(t.shape, device=DEV, generator=g) * 0.3
                t.copy_(A.to_fp8(x.bfloat16()) if kv else x)
        need = [(c + n + 31) // 32 for c, n in zip(prefix, new)]
        bt = np.zeros((rows, max(need)), np.int32)
        at = 0
        for b, k in enumerate(need):
            bt[b, :k] = np.arange(at, at + k)
            at += k
        pos = np.concatenate([np.arange(c, c + n) for c, n in zip(prefix, new)]).astype(np.int32)
        row = np.repeat(np.arange(rows), new)
        cu_q = np.concatenate([[0], np.cumsum(new)]).astype(np.int32)
        cu_k = np.concatenate([[0], np.cumsum(np.add(prefix, new))]).astype(np.int32)
        ids = np.random.RandomState(0).randint(0, 512, sum(new)).astype(np.int32)
        plan = dict(input_ids=ids, positions=pos, slot_mapping=bt[row, pos // 32].astype(np.int64) * 32 + pos % 32,
                    cu_q=cu_q, cu_k=cu_k, max_q=max(new), has_prefix=max(prefix) > 0, block_tables=bt,
                    req_ids=np.arange(rows), temperature=np.zeros(rows, np.float32), top_p=np.ones(rows, np.float32),
                    top_k=np.full(rows, 1 << 30), sample=np.ones(rows, np.int32), logit_rows=cu_q[1:].astype(np.int64) - 1)
        r.prefill(plan)
        assert r.kept_logits.dtype == torch.float32
        out.append((r.kept_logits.clone(), [t.float().clone() for pair in r.kv for t in pair]))
    (a, ca), (b, cb) = out
    # two roundings of the same sums: three layers of bf16 steps (2^-8) on logits of size one
    assert float((a - b).abs().max()) < 0.06 * max(1.0, float(a.abs().max()))
    step = 2.0 ** -3 if kv else 2.0 ** -6  # a step of the cache's type, a few roundings apart
    for x, y in zip(ca, cb):
        assert bool(((x - y).abs() <= 0.05 + step * x.abs()).all())


@pytest.mark.parametrize("rows", [1, 24, 64, 65, 96])
@pytest.mark.parametrize("K", [512, 896, 1536, 4096])
def test_scoring_head(rows, K):
    """fp32 logits from the matrix cores: no further from double precision than the fp32 library product."""
    from types import SimpleNamespace

    from areal_vllm_amd.inference.model_runner import ModelRunner

    g = torch.Generator(device=DEV).manual_seed(rows + K)
    x = torch.randn(rows, K, device=DEV, generator=g).bfloat16()
    w = (torch.randn(4096 + 32, K, device=DEV, generator=g) * 0.02).bfloat16()
    runner = SimpleNamespace(model=SimpleNamespace(head_weight=w), LM_HEAD_OWN_MAX_ROWS=ModelRunner.LM_HEAD_OWN_MAX_ROWS)
    runner._lm_head_own = lambda y: ModelRunner._lm_head_own(runner, y)
    got = ModelRunner._lm_head(runner, x, fp32=True)
    assert got.dtype == torch.float32
    want = x.double() @ w.double().t()
    lib = torch.nn.functional.linear(x.float(), w.float())
    rms = lambda y: float((y.double() - want).pow(2).mean()) ** 0.5
    assert rms(got) <= rms(lib)
