"""Decode projections of a few rows against the same arithmetic in fp64 with the same rounding points, and the five-launch
layer inside the runner against the split-K layer."""
import math

import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.ops import decode_skinny as sk

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


def _norm(h, w, gemma):
    x = h.double() * torch.rsqrt(h.double().pow(2).mean(-1, keepdim=True) + 1e-6) * (w.double() + (1.0 if gemma else 0.0))
    return x.bfloat16().double()


def _close(got, want, bits=7):
    # two correctly rounded bf16 values of sums that differ in the last fp32 bits, or products of two such: a few 2^-8
    err = (got.double() - want).abs() - 2.0 ** -bits * want.abs()
    assert float(err.max()) < 2.0 ** -bits * float(want[want != 0].abs().mean()), float(err.max())


@pytest.mark.parametrize("M", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("N,K", [(1536, 1536), (1536, 8960), (3584, 18944), (7, 64), (40, 25600), (300, 576), (5000, 1024)])
def test_linear_residual(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M * 7 + N)
    x = torch.randn(M + 1, K + 8, device=DEV, generator=g).bfloat16()[:M, :K]  # rows further apart than they are long
    w = (torch.randn(N, K, device=DEV, generator=g) / math.sqrt(K)).bfloat16()
    r = torch.randn(M, N, device=DEV, generator=g).bfloat16()
    y = x.double() @ w.double().t()
    _close(sk.linear_residual(x, w), y)
    got = sk.linear_residual(x, w, r)
    _close(got, y.bfloat16().double() + r.double())
    assert torch.equal(got, sk.linear_residual(x, w, r))


@pytest.mark.parametrize("M", [1, 2, 4, 7, 8])
@pytest.mark.parametrize("F,K", [(8960, 1536), (100, 64), (4096, 1024), (11008, 2048), (18944, 3584), (14336, 4096), (36, 8192)])
@pytest.mark.parametrize("gemma,act", [(False, "silu"), (True, "gelu_tanh")])
def test_norm_gated(M, F, K, gemma, act):
    g = torch.Generator(device=DEV).manual_seed(M * 7 + F)
    h = torch.randn(M, K, device=DEV, generator=g).bfloat16() * 3
    nw = torch.rand(K, device=DEV, generator=g).bfloat16() + 0.5
    w = (torch.randn(2 * F, K, device=DEV, generator=g) / math.sqrt(K)).bfloat16()
    y = (_norm(h, nw, gemma) @ w.double().t()).bfloat16().double()
    gate = torch.nn.functional.silu(y[:, :F]) if act == "silu" else torch.nn.functional.gelu(y[:, :F], approximate="tanh")
    # gate and up are rounded before they are multiplied: two values next to a rounding edge may each be off by one step
    _close(sk.norm_gated(h, nw, w, eps=1e-6, gemma=gemma, act=act), gate * y[:, F:], bits=6)


@pytest.mark.parametrize("M", [1, 2, 4, 8])
@pytest.mark.parametrize("Hq,Hkv,D,K,fp8", [(12, 2, 128, 1536, False), (12, 2, 128, 1536, True), (28, 4, 128, 3584, False),
                                            (2, 1, 64, 192, False), (8, 1, 256, 2048, True), (3, 3, 16, 64, False)])
@pytest.mark.parametrize("with_bias", [True, False])
def test_norm_qkv_rope(M, Hq, Hkv, D, K, fp8, with_bias):
    g = torch.Generator(device=DEV).manual_seed(M * 7 + K)
    h = torch.randn(M, K, device=DEV, generator=g).bfloat16()
    nw = torch.rand(K, device=DEV, generator=g).bfloat16() + 0.5
    N = (Hq + 2 * Hkv) * D
    w = (torch.randn(N, K, device=DEV, generator=g) / math.sqrt(K)).bfloat16()
    bias = torch.randn(N, device=DEV, generator=g).bfloat16() if with_bias else None
    pos = torch.randint(0, 500, (M,), device=DEV, generator=g, dtype=torch.int32)
    slots = (torch.randperm(40 * 32, device=DEV, generator=g)[:M]).long()
    if M > 1:
        slots[1] = -1  # a retired row: nothing is written
    tab = ops.RotaryTable(D, 512, 1e4, DEV)
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
    caches = [ops.alloc_kv_cache(40, Hkv, D, dt, DEV) for _ in range(2)]
    q = sk.norm_qkv_rope(h, nw, w, bias, pos, slots, tab, *caches[0], Hq, Hkv, D, eps=1e-6)
    y = _norm(h, nw, False) @ w.double().t()
    if with_bias:
        y = y + bias.double()
    want = y.bfloat16().view(M, Hq + 2 * Hkv, D).contiguous()
    ops.rope_and_cache_write_(want, pos, slots, tab, *caches[1], Hq, Hkv)
    # a rotated value holds its partner's rounding too, whatever its own size: one step of values below 8 is 2^-5
    _close(q, want[:, :Hq].double(), bits=5)
    for a, b in zip(*caches):  # fp8: a value next to a rounding edge of 3 bits of mantissa may take the other one
        _close(a.float(), b.float().double(), bits=2 if fp8 else 5)
        assert torch.equal(a.float() != 0, b.float() != 0) or float(((a.float() != 0) != (b.float() != 0)).sum()) < 3


@pytest.mark.parametrize("M", [1, 2])
@pytest.mark.parametrize("N,K", [(2000, 1600), (256, 3072), (5000, 3136), (1536, 6144), (260, 12288), (7, 12352)])
def test_linear_residual_of_every_split_of_the_waves(M, N, K):
    """Two, four and eight waves along K, first and last depth of each; one weight row a wave and many; a last workgroup of few."""
    test_linear_residual(M, N, K)


@pytest.mark.parametrize("M", [3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("N,K", [(2048, 3136), (2049, 3136), (1025, 6144), (9, 6208), (2048, 12288), (7, 12352), (896, 3072)])
def test_linear_residual_of_more_rows_by_dot_products(M, N, K):
    """Either side of the columns and depths that they are taken for; four and eight waves along K and more than one turn of them."""
    test_linear_residual(M, N, K)


@pytest.mark.parametrize("M", [1, 2])
@pytest.mark.parametrize("Hq,Hkv,D,K", [(40, 8, 128, 2048), (2, 1, 128, 8192), (6, 2, 48, 3136), (2, 2, 16, 12288)])
def test_norm_qkv_rope_of_every_split_of_the_waves(M, Hq, Hkv, D, K):
    test_norm_qkv_rope(M, Hq, Hkv, D, K, False, True)


@pytest.mark.parametrize("rows,hidden,inner,heads,extra", [
    (1, 256, 512, (4, 2, 64), dict(family="qwen2", qkv_bias=True)), (2, 1536, 1024, (12, 2, 128), dict(family="qwen2", qkv_bias=True)),
    (3, 256, 576, (4, 2, 128), dict(family="llama")), (6, 1536, 1024, (12, 2, 128), dict(family="qwen2", qkv_bias=True)),
    (6, 256, 512, (2, 1, 256), dict(family="gemma", hidden_act="gelu_tanh", gemma_norm=True)),
    (1, 2048, 1024, (16, 2, 128), dict(family="llama")), (2, 4096, 512, (8, 8, 128), dict(family="qwen2", qkv_bias=True))])
@pytest.mark.parametrize("fp8", [False, True])
def test_layer_inside_the_runner(rows, hidden, inner, heads, extra, fp8):
    """Captured decode plans of several steps on the five-launch layer and on split-K GEMMs with row kernels: logits, tokens and
    what is written into the cache."""
    import numpy as np

    from areal_vllm_amd.inference.model_runner import ModelRunner
    from areal_vllm_amd.models.config import ModelConfig
    from areal_vllm_amd.models.transformer import Transformer

    hq, hkv, D = heads
    cfg = ModelConfig(vocab_size=512, hidden_size=hidden, n_layers=3, n_q_heads=hq, n_kv_heads=hkv, head_dim=D, intermediate_size=inner,
                      max_position_embeddings=2048, tie_word_embeddings=True, **extra)
    model = Transformer(cfg, dtype=torch.bfloat16, device=torch.device(DEV))
    model.requires_grad_(False)
    model.eval()
    model.flatten()
    g = torch.Generator(device=DEV).manual_seed(hidden + rows)
    with torch.no_grad():
        for n, p in model.named_parameters():
            x = torch.randn(p.shape, device=DEV, generator=g)
            if n == "embed":  # large beside what a layer adds: every row's next token is its own, whatever is rounded how
                p.copy_(x * 0.5)
            elif p.dim() > 1:
                p.copy_(x * 0.5 / p.shape[1] ** 0.5)
            else:
                p.copy_(x * 0.1 + (0.0 if "bias" in n or extra.get("gemma_norm") else 1.0))
    steps, ctx = 4, [5 + 61 * b for b in range(rows)]
    width = (max(ctx) + steps) // 32 + 1
    table = (np.random.RandomState(0).permutation(rows * width) + 1).reshape(rows, width).astype(np.int32)
    pos = np.asarray(ctx, np.int32)
    plan = dict(req_ids=list(range(rows)), temperature=np.zeros(rows, np.float32), top_p=np.ones(rows, np.float32),
                top_k=np.full(rows, 1 << 30, np.int64), n_steps=steps, input_ids=np.arange(rows, dtype=np.int32) * 7 + 3, positions=pos,
                context_lens=pos + 1, block_tables=table, max_pages=width,
                slot_mapping=table[np.arange(rows), pos // 32].astype(np.int64) * 32 + pos % 32)
    got = []
    for five in (False, True):
        r = ModelRunner(model, rows * width + 1, width * 32, rows, decode_steps=steps, buckets=[rows],
                        **(dict(kv_dtype=torch.float8_e4m3fn) if fp8 else {}))
        if not five:
            r.SKINNY_MAX_ROWS = r.SKINNY_MAX_ROWS_WIDE = 0
        assert r._skinny(rows) == five
        gen = torch.Generator(device=DEV).manual_seed(1)
        for pair in r.kv:
            for t in pair:
                t.copy_((torch.randn(t.shape, device=DEV, generator=gen) * 0.5).to(t.dtype))
        r.keep_logits = True
        for _ in range(2):  # captured by the first plan, replayed by the second
            tokens, _ = r.decode(plan)
        got.append((tokens.copy(), r.static[rows]["logits"].clone(), [t.float().clone() for pair in r.kv for t in pair]))
    (ta, la, ca), (tb, lb, cb) = got
    assert np.array_equal(ta, tb) and np.array_equal(ta[:, :rows], np.tile(plan["input_ids"], (steps, 1)))
    # the same rounding points, sums in another order: three layers of bf16 steps (2^-8), as between the prefill's two layers
    assert float((la - lb).abs().max()) < 0.06 * max(1.0, float(la.abs().max()))
    step = 2.0 ** -3 if fp8 else 2.0 ** -6  # a step of the cache's type, a few roundings apart
    for x, y in zip(ca, cb):
        assert bool(((x - y).abs() <= 0.05 + step * x.abs()).all())


@pytest.mark.parametrize("M", [1, 2, 5])
def test_rotation_roundings(M):
    """Which product of a rotated value is rounded by itself: lo c - r(hi s), hi c + r(lo s), bit for bit, and so the results of every decode
    step. The projection is exact: rows of +-1 with a mean square of one, weights in sixteenths."""
    Hq, Hkv, D, K = 60, 2, 128, 512
    ones, tab = torch.ones(K, device=DEV).bfloat16(), ops.RotaryTable(D, 4096, 1e6, DEV)
    for seed in range(40):
        g = torch.Generator(device=DEV).manual_seed(seed * 8 + M)
        x = (torch.randint(0, 2, (M, K), device=DEV, generator=g) * 2 - 1).bfloat16()
        w = (torch.randint(-9, 10, ((Hq + 2 * Hkv) * D, K), device=DEV, generator=g) / 16).bfloat16()
        pos = torch.randint(0, 4096, (M,), device=DEV, generator=g, dtype=torch.int32)
        kc, vc = ops.alloc_kv_cache(1, Hkv, D, torch.bfloat16, DEV)
        q = sk.norm_qkv_rope(x, ones, w, None, pos, torch.full((M,), -1, device=DEV).long(), tab, kc, vc, Hq, Hkv, D, eps=0.0)
        y = (x.float() @ w.float().t()).bfloat16().float()[:, :Hq * D].view(M, Hq, 2, D // 2)
        lo, hi = y[:, :, 0], y[:, :, 1]
        c, s = (t[pos.long()][:, None] for t in (tab.cos, tab.sin))
        want = torch.cat([lo.double() * c.double() - (hi * s).double(), hi.double() * c.double() + (lo * s).double()], -1)
        assert torch.equal(q, want.float().bfloat16()), int((q != want.float().bfloat16()).sum())
