"""The activation of the gated product's epilogue over all gates that bf16 holds."""
import pytest
import torch

from areal_vllm_amd.ops import train_gemm as tg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("up", [1.0, -1.5])
def test_every_gate(up):
    gates = torch.arange(1 << 16, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).cuda()
    F, K = gates.numel(), 128
    w = torch.zeros(2 * F, K, device="cuda", dtype=torch.bfloat16)
    w[:F, 0], w[F:, 1] = gates, up
    x = torch.zeros(3, K, device="cuda", dtype=torch.bfloat16)
    x[:, :2] = 1.0  # one product a gate, with 1: exact
    out = tg.tgemm_swiglu(x, w)
    assert torch.equal(out[0].view(torch.int16), out[2].view(torch.int16))
    g, got = gates.double(), out[0].double()
    want = g * torch.sigmoid(g) * up
    assert got[g == float("inf")].tolist() == [up * float("inf")]
    assert got[g.isnan() | (g == -float("inf"))].isnan().all()
    # where the exponential is finite: one rounding to bf16 (half a step is at most 2^-8 of the value), an exponential whose
    # argument of up to 89 was rounded to 24 bits, and bf16's subnormal numbers kept or not
    sure = (g > -88.7) & g.isfinite() & (want.abs() < 3.3e38)
    assert ((got - want)[sure].abs() <= want[sure].abs() * (2.0 ** -8 + 2.0 ** -15) + 2.0 ** -126).all()
    assert got[(g < -89) & g.isfinite()].eq(0).all()
