"""Unfiltered sampler: the first of equal keys, groups of eight that are forbidden as a whole, rows off the 16-byte grid."""
import pytest
import torch

from areal_vllm_amd import ops

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [5, 8, 63, 1003, 4096, 50257, 151936])
@pytest.mark.parametrize("B", [1, 3, 130])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_first_of_equal(V, B, dtype):
    g = torch.Generator(device=DEV).manual_seed(V + B)
    logits = torch.randint(-3, 4, (B, V), device=DEV, generator=g).to(dtype)  # hundreds of equal maxima
    logits[:, : V // 3] = -float("inf")
    step = torch.zeros(1, dtype=torch.int64, device=DEV)
    tok, lp = ops.sample(logits, torch.zeros(B, device=DEV), None, None, 7, step)
    top = logits.float().max(-1, keepdim=True).values
    want = (logits.float() == top).int().argmax(-1)
    assert torch.equal(tok, want)
    full = torch.log_softmax(logits.double(), -1).gather(1, want[:, None])[:, 0]
    # fp32 sums of up to 151936 exponentials between e^-6 and 1
    assert float((lp.double() - full).abs().max()) < 1e-4
    # at temperature 1 a forbidden entry is never drawn
    tok, lp = ops.sample(logits, torch.ones(B, device=DEV), None, None, 7, step)
    assert bool((tok >= V // 3).all()) and bool(torch.isfinite(lp).all())
