"""Grouped products whose weights are read past the caches, and those whose weights are not: the same bits."""
import pytest
import torch

from areal_vllm_amd.ops.grouped_gemm import _launch

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,K,N", [(8, 128, 4352), (40, 192, 832), (300, 64, 128)])
def test_same_bits(E, K, N):
    g = torch.Generator().manual_seed(E)
    w = (torch.randn(E, N, K, generator=g) / K ** 0.5).bfloat16().to(DEV)
    full = torch.randint(0, 100, (E,), generator=g)
    full[0], full[-1] = 0, 127
    x = torch.randn(int(full.sum()), K, generator=g).bfloat16().to(DEV)
    first = torch.cat([torch.zeros(1, dtype=torch.long), full.cumsum(0)[:-1]])

    def run(counts):
        rows = torch.cat([torch.arange(f, f + c) for f, c in zip(first.tolist(), counts.tolist())])
        off = torch.cat([torch.zeros(1, dtype=torch.long), counts.cumsum(0)]).int().to(DEV)
        return rows, _launch(x[rows.to(DEV)].contiguous(), w, off)

    # few rows, one an expert (more than 256 workgroups), up to and over 48 an expert, all of them
    cases = [run(c) for c in (full.clamp(max=1) * (torch.arange(E) < 2), full.clamp(max=1), full.clamp(max=47), full)]
    rows, y = cases[-1]
    expert = torch.repeat_interleave(torch.arange(E), full).to(DEV)
    for e in range(0, E, max(1, E // 8)):
        at = expert == e
        want = x[at].float() @ w[e].float().t()
        # bf16 of sums of size one over at most 192 products: one rounding
        assert bool(((y[at].float() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())
    for rows, z in cases[:-1]:
        assert torch.equal(z, y[rows.to(DEV)])
