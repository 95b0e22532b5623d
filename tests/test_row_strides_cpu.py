"""Row strides that 32-bit offsets do not reach are refused, on the host, before any launch."""
from types import SimpleNamespace

import pytest
import torch

from areal_vllm_amd.ops import _lib as L
from areal_vllm_amd.ops import train_gemm as tg

pytestmark = pytest.mark.skipif(not L.available(), reason="the kernel library is not built")


def _operand(rows, cols, stride):
    return SimpleNamespace(is_cuda=True, dtype=torch.bfloat16, dim=lambda: 2, shape=(rows, cols), stride=lambda i: (stride, 1)[i],
                           data_ptr=lambda: 1 << 20)


@pytest.mark.parametrize("ldy,ldx,taken", [(128, 256, True), (1 << 24, 1 << 24, True), ((1 << 24) + 8, 256, False),
                                           (128, (1 << 24) + 8, False), (1 << 25, 1 << 25, False)])
def test_row_strides(ldy, ldx, taken):
    acc = SimpleNamespace(dtype=torch.float32, shape=(128, 256), stride=lambda i: (256, 1)[i])
    assert tg.wgrad_supported(_operand(1024, 128, ldy), _operand(1024, 256, ldx), acc) == taken
    if not taken:
        p = L.c_void_p(1 << 20)  # never read: the entry refuses the strides first
        assert L.lib().areal_tgemm_wgrad(p, L.c_int64(ldy), p, L.c_int64(ldx), p, L.c_int64(256), L.c_int(1024), L.c_int(128),
                                         L.c_int(256), L.c_int(1), L.c_int(1), L.c_void_p(0), L.c_void_p(0)) == -1


@pytest.mark.parametrize("which", range(4))
def test_flash_row_strides(which):
    p, far = L.c_void_p(1 << 20), (1 << 24) + 8
    st = [L.c_int64(far if i == which else 1536) for i in range(4)]  # q, k, v, dO
    i, one, scale = L.c_int, L.c_int64(1536), L.c_float(1.0)
    if which in (1, 2):  # the forward stages keys and values
        assert L.lib().areal_flash_fwd(p, p, p, p, p, p, p, i(1), i(64), i(64), i(12), i(2), i(128), *st[:3], one, scale, i(1),
                                       L.c_void_p(0)) == -5
    assert L.lib().areal_flash_bwd(p, p, p, p, p, p, p, p, p, p, p, i(1), p, p, i(1), i(64), i(64), i(64), L.c_int64(64), i(12),
                                   i(2), i(128), *st[:3], one, st[3], one, one, one, scale, i(1), L.c_void_p(0)) == -5


def test_far_rows_are_copied():
    from areal_vllm_amd.ops.attention import _near_rows

    t = torch.arange(24.).view(3, 2, 4)
    assert _near_rows(t) is t
    far = torch.arange(8.).as_strided((1, 2, 4), ((1 << 24) + 8, 4, 1))
    near = _near_rows(far)
    assert near.stride(0) == 8 and torch.equal(near, far)
