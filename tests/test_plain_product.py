"""`linear` without gradients under what rewrites or records ATen calls: the own product, which works on raw pointers, steps aside."""
import pytest
import torch
import torch.nn.functional as F
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.autograd import forward_ad
from torch.utils.flop_counter import FlopCounterMode

from areal_vllm_amd import ops
from areal_vllm_amd.ops import train_gemm as tg


def _seen(call, *args):
    """plain() of the operands as `call` sees them."""
    seen = []

    def f(x, w):
        seen.append(tg.plain(x, w))
        return F.linear(x, w)

    call(f, *args)
    return seen


def test_what_is_plain():
    x, w = torch.randn(3, 8), torch.nn.Parameter(torch.randn(4, 8))
    with torch.no_grad():
        assert _seen(lambda f: f(x, w)) == [True]
        assert _seen(lambda f: torch.vmap(f, (0, None))(torch.randn(2, 3, 8), w)) == [False]
        assert False in _seen(lambda f: torch.jit.trace(f, (x, w.detach())))
        with forward_ad.dual_level():
            assert tg.plain(x, w) and not tg.plain(forward_ad.make_dual(x, x), w) and not tg.plain(x, forward_ad.make_dual(w, w))
        with FlopCounterMode(display=False):
            assert not tg.plain(x, w)
        with FakeTensorMode() as mode:
            fake = mode.from_tensor(x)
        assert not tg.plain(fake, w)
        with torch.autocast("cpu", torch.bfloat16):
            assert not tg.plain(x, w)


@pytest.mark.gpu
def test_own_product_steps_aside():
    torch.manual_seed(0)
    x, w = torch.randn(2, 700, 16384, device="cuda").bfloat16(), (torch.randn(64, 16384, device="cuda") / 128).bfloat16()
    assert tg._forward_own(700, 16384, 64)
    # both products round sums of size one once: half a step of bf16 on either side
    same = lambda a, b: torch.allclose(a.double(), b.double(), rtol=2.0 ** -7, atol=1e-3)
    with torch.no_grad():
        want = F.linear(x, w)
        assert same(ops.linear(x[0], w), want[0])
        assert same(torch.vmap(ops.linear, (0, None))(x, w), want)
        traced = torch.jit.trace(lambda t: ops.linear(t, w), x[0], check_trace=False)
        assert same(traced(x[1]), want[1])
        with forward_ad.dual_level():
            tangent = forward_ad.unpack_dual(ops.linear(forward_ad.make_dual(x[0], x[1]), w)).tangent
            assert tangent is not None and same(tangent, want[1])
        with torch.autocast("cuda", torch.float16):
            assert ops.linear(x[0], w).dtype == torch.float16
        with FlopCounterMode(display=False) as count:
            ops.linear(x[0], w)
        assert count.get_total_flops() == 2 * 700 * 16384 * 64
