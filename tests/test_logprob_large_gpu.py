"""Log-probabilities over logits that are read past the caches (256 MB and more) and of the next smaller number of rows."""
import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype,V", [(torch.bfloat16, 65536), (torch.bfloat16, 65541), (torch.float32, 32768), (torch.float32, 32769)])
@pytest.mark.parametrize("more", [-1, 0, 1])
def test_both_sides_of_the_line(dtype, V, more):
    lp = importlib.import_module("areal_vllm_amd.ops.logprob")
    ld = -(-V // 8) * 8
    T = (256 << 20) // (ld * dtype.itemsize) + more + (ld != V)
    g = torch.Generator(device=DEV).manual_seed(V)
    buf = torch.randn(T, ld, device=DEV, generator=g, dtype=torch.float32).mul_(2).to(dtype)
    z = buf[:, :V]
    lab = torch.randint(V, (T,), device=DEV, generator=g)
    dl, de = torch.randn(T, device=DEV, generator=g), torch.randn(T, device=DEV, generator=g)
    logp, ent, lse, ez = lp._fwd(z, lab, 1.0)
    rows = torch.tensor([0, T // 2, T - 1], device=DEV)
    x = z[rows].double().requires_grad_(True)
    ls = torch.log_softmax(x, -1)
    want_lp, want_ent = ls.gather(1, lab[rows, None])[:, 0], -(ls.exp() * ls).sum(-1)
    (want_lp * dl[rows].double() + want_ent * de[rows].double()).sum().backward()
    # sums of 2^15 fp32 values of one sign: a few 2^-24 of a logarithm near 12
    assert (logp[rows].double() - want_lp).abs().max() < 2e-5 and (ent[rows].double() - want_ent).abs().max() < 2e-4
    pad = buf[:, V:].clone()
    got = lp._bwd_inplace(z, lab, 1.0, lse, ez, dl, de)[rows].double()
    # bf16: rounded once
    assert (got - x.grad).norm() / x.grad.norm() < (4e-3 if dtype == torch.bfloat16 else 1e-5)
    assert torch.equal(buf[:, V:], pad)
