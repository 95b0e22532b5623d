"""Row strides that the weight-gradient GEMM's 32-bit offsets do not reach are refused, on the host, before any launch."""
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
                                         L.c_int(256), L.c_int(0), L.c_int(1), L.c_void_p(0)) == -1
