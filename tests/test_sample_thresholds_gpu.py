"""Top-k and top-p sets of the sampler against sorted rows in double precision, over row shapes that fill its histograms
unevenly: constant, flat, one far entry on either side, masked entries, wide and narrow ranges."""
import pytest
import torch

from areal_vllm_amd import ops

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


def _rows(V, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    r = torch.randn(V, generator=g)
    rows = [r, 3 * r, 12 * r, 0.01 * r, torch.full((V,), 1.5), r.sign(), 1e-30 * r]
    for at, v in ((V // 2, 40.), (V // 3, -3e4), (V // 4, float("-inf"))):
        x = r.clone()
        x[at] = v
        rows.append(x)
    x = r.clone()
    x[torch.rand(V, generator=g) < 0.9] = float("-inf")  # nine in ten masked
    x[-1] = r[-1]
    rows.append(x)
    x = torch.full((V,), -1e9)
    x[: max(2, V // 50)] = r[: max(2, V // 50)]
    rows.append(x)
    return torch.stack(rows).to(dtype)


@pytest.mark.parametrize("V", [3, 37, 1024, 4097, 32000, 151936])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("k,p", [(0, 0.0), (0, 0.1), (0, 0.9), (0, 0.9999), (1, 1.0), (2, 1.0), (50, 0.7), (300, 1.0),
                                 (5000, 1.0), (5000, 0.95), (100000, 1.0)])
@pytest.mark.parametrize("temp", [1.0, 0.05, 3.0])
def test_sets(V, dtype, k, p, temp):
    logits = _rows(V, dtype, V + k).to(DEV)
    B = logits.shape[0]
    t = torch.full((B,), temp, device=DEV)
    kk = torch.full((B,), k if k else V, dtype=torch.int32, device=DEV)
    pp = torch.full((B,), p, device=DEV)
    z = (logits.float() * (1.0 / t)[:, None])
    s, order = z.double().sort(dim=1, descending=True)
    if 1 <= k < V:
        kth = s[:, k - 1:k]
        in_k = z.double() >= kth
    else:
        in_k = torch.ones_like(z, dtype=torch.bool)
    prob = torch.where(in_k, (z.double() - s[:, :1]).exp(), 0.0)
    prob = prob / prob.sum(1, keepdim=True)
    # mass strictly above an entry: it belongs to the set as long as that falls short of p
    ps = prob.gather(1, order)
    above_sorted = ps.cumsum(1) - ps
    first = torch.searchsorted(-s, -s, right=False)  # ties share the position of the first of them
    above = torch.empty_like(prob).scatter_(1, order, above_sorted.gather(1, first))
    eps = 2e-5  # the sums over V <= 2^18 fp32 exponentials and 2^-40 steps differ from these by less
    wide, sure = in_k & (above < p + eps), in_k & (above < p - eps)
    sure.scatter_(1, order[:, :1], True)
    if p >= 1.0:
        wide, sure = in_k, in_k
    for step in range(6):
        st = torch.full((1,), step, dtype=torch.int64, device=DEV)
        free = ops.sample(logits, t, None, None, 7, st.clone())[0]
        tok, lp = ops.sample(logits, t, kk, pp, 7, st.clone())
        assert bool(wide.gather(1, tok[:, None]).all())
        hit = sure.gather(1, free[:, None])[:, 0]  # the same noise: a free draw that lies in the set is the filtered one
        assert torch.equal(tok[hit], free[hit])
        want = torch.log_softmax(z, 1).gather(1, tok[:, None])[:, 0]
        assert torch.allclose(lp, want, atol=2e-3, rtol=1e-5)
