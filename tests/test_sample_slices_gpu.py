"""Filtered sampling with the rows split over workgroups against one workgroup a row: the same tokens and counts."""
import math
import sys

import pytest
import torch

from areal_vllm_amd import ops

S = sys.modules["areal_vllm_amd.ops.sampling"]
DEV = "cuda:0"
pytestmark = pytest.mark.gpu


# rows that fill a slice's histogram unevenly, limits around the largest k that is handed on, more rows than slices
@pytest.mark.parametrize("V", [100, 4096, 20001])
@pytest.mark.parametrize("B", [1, 12, 300])
@pytest.mark.parametrize("k", [1, 127, 128, 129])
@pytest.mark.parametrize("p", [1.0, 0.6])
def test_same_as_one_workgroup(V, B, k, p, monkeypatch):
    g = torch.Generator().manual_seed(V + B + k)
    logits = 3 * torch.randn(B, V, generator=g)
    for b in range(B):
        if b % 6 == 1:
            logits[b] = 1.5  # all equal: too many for a slice
        elif b % 6 == 2:
            logits[b] = logits[b].sort().values  # the largest in one slice
        elif b % 6 == 3:
            logits[b, torch.rand(V, generator=g) < 0.99] = float("-inf")
            logits[b, V - 1] = 0.0
        elif b % 6 == 4:
            logits[b, V // 2] = 60.0
    logits = logits.bfloat16().to(DEV)
    t = (0.5 + torch.rand(B, generator=g)).to(DEV)
    t[B // 2] = 0.0 if B > 1 else t[0]  # greedy
    kk = torch.full((B,), k, dtype=torch.int32, device=DEV)
    kk[B // 3] = k if B == 1 else V
    pp = torch.full((B,), p, device=DEV)
    active = torch.ones(B, dtype=torch.int32, device=DEV)
    active[0] = int(B == 1)  # the workgroup that counts the step on
    slot = torch.full((B,), -1, dtype=torch.int32, device=DEV)
    slot[: min(B, 3)] = torch.arange(min(B, 3), dtype=torch.int32, device=DEV)
    pen = torch.full((B,), 0.7, device=DEV)
    got = []
    monkeypatch.setattr(S, "_slices", lambda B, V: min(16, -(-512 // B)))
    for most in (0, 384):
        monkeypatch.setattr(S, "SPLIT_FILTERED_MAX_ROWS", most)
        counts = ops.TokenCounts(3, V, torch.device(DEV))
        step = torch.zeros(1, dtype=torch.int64, device=DEV)
        out = [ops.sample(logits, t, kk, pp, 11, step, active=active, counts=counts, count_slot=slot, freq_pen=pen,
                          pres_pen=pen) for _ in range(3)]
        assert int(step) == 3
        got.append((torch.stack([o[0] for o in out]), torch.stack([o[1] for o in out]), counts.table.clone()))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][2], got[1][2])
    # sums of V fp32 exponentials in another order
    assert torch.allclose(got[0][1], got[1][1], atol=1e-4, rtol=1e-5)


# the rule's own counts; rows of an odd length start off the 16-byte grid and are walked entry by entry, by all slices
@pytest.mark.parametrize("B,V,n", [(3, 50257, 6), (70, 50257, 6), (200, 50257, 2), (300, 50257, 3), (350, 50257, 1), (64, 65536, 8)])
@pytest.mark.parametrize("k,p", [(50, 0.95), (1 << 30, 0.9), (200, 1.0)])
def test_the_rule(B, V, n, k, p, monkeypatch):
    assert S._slices(B, V) == n
    torch.manual_seed(B)
    logits = 3 * torch.randn(B, V, device=DEV)
    t, kk, pp = torch.ones(B, device=DEV), torch.full((B,), k, dtype=torch.int32, device=DEV), torch.full((B,), p, device=DEV)
    got = [ops.sample(logits, t, kk, pp, 5, torch.zeros(1, dtype=torch.int64, device=DEV))]
    monkeypatch.setattr(S, "SPLIT_FILTERED_MAX_ROWS", 0)
    got.append(ops.sample(logits, t, kk, pp, 5, torch.zeros(1, dtype=torch.int64, device=DEV)))
    assert torch.equal(got[0][0], got[1][0])
    assert torch.allclose(got[0][1], got[1][1], atol=1e-4, rtol=1e-5)  # as above


@pytest.mark.parametrize("B,V", [(1, 8), (3, 517), (64, 4097), (65, 40000), (1100, 300)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_unfiltered_rows_whose_slices_are_mostly_masked(B, V, dtype):
    """Slices of one row without a finite entry, and rows with a single one (its log-prob is zero) in any of them."""
    g = torch.Generator(device="cuda").manual_seed(B)
    logits = torch.full((B, V), -math.inf, dtype=dtype, device="cuda")
    at = torch.randint(V, (B,), generator=g, device="cuda")
    logits[torch.arange(B, device="cuda"), at] = 3.0
    step = torch.zeros(1, dtype=torch.int64, device="cuda")
    tok, lp = ops.sample(logits, torch.full((B,), 0.9, device="cuda"), None, None, seed=5, step=step)
    assert torch.equal(tok, at) and float(lp.abs().max()) < 1e-6 and step.item() == 1
