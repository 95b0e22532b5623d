"""The gated decode projection on every tile that it has: ragged rows, a narrower last range, one step and many, rings of all depths."""
import pytest
import torch

from areal_vllm_amd.ops import _lib as L

pytestmark = pytest.mark.gpu


def _sixteenths(*shape):
    """Sums of their products are exact in fp32, in any order."""
    return (torch.randint(-8, 9, shape, device="cuda") / 16).bfloat16()


@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("ct", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("rt", [1, 2, 3, 4, 5, 6, 7, 8])
def test_every_tile(rt, ct, act):
    torch.manual_seed(rt * 10 + ct)
    for mblocks in (1, 2, 3, 4):
        w, steps, stages = 16 * ct - (0, 4, 8, 12)[(mblocks + rt) % 4], (1, 2, 5, 9)[(mblocks + ct) % 4], 2 + (mblocks + rt + ct) % 5
        M, F, K = 32 * rt * mblocks - 13, 3 * w + (4 if w > 4 else 0), 64 * steps
        x, wt = _sixteenths(M, K + 8)[:, :K], _sixteenths(2 * F, K)
        y = torch.full((M + 2, F + 8), float("nan"), dtype=torch.bfloat16, device="cuda")
        rc = L.lib().areal_dswiglu(L.ptr(x), L.c_int64(K + 8), L.ptr(wt), L.ptr(y), L.c_int64(F + 8), *[L.c_int(v) for v in (
            M, F, K, w, mblocks, stages, mblocks & 1, act)], L.stream_ptr())
        assert rc == 0
        g, u = (x.float() @ wt.float().t()).bfloat16().double().split(F, 1)
        want = u * (torch.nn.functional.gelu(g, approximate="tanh") if act else g * torch.sigmoid(g))
        err = (y[:M, :F].double() - want).abs()
        # one rounding to bf16 (half a step is at most 2^-8 of the value), fp32 arithmetic in front of it; GELU's 1 + tanh cancels for
        # negative gates: 2^-22 of the gate
        assert (err <= want.abs() * (2.0 ** -8 + 2.0 ** -14) + act * (g * u).abs() * 2.0 ** -22 + 1e-30).all(), (mblocks, float(err.max()))
        assert y[M:].isnan().all() and y[:, F:].isnan().all()
