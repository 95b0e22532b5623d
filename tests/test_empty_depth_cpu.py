"""Products over no columns at all (K = 0) are not for the kernels, whose first loads do not ask: the rules leave them to the
library, the C entries refuse them ahead of any launch."""
from types import SimpleNamespace

import pytest
import torch

from areal_vllm_amd.ops import _lib as L
from areal_vllm_amd.ops import decode_gemm as dg
from areal_vllm_amd.ops import train_gemm as tg
from areal_vllm_amd.ops.grouped_gemm import _hip_ok


def _operand(*shape):
    return SimpleNamespace(is_cuda=True, dtype=torch.bfloat16, dim=lambda: len(shape), shape=shape, data_ptr=lambda: 1 << 20,
                           stride=lambda i: shape[-1] if i < len(shape) - 1 else 1, is_contiguous=lambda: True)


@pytest.mark.parametrize("K", [128, 0])
def test_rules(K):
    x, w = _operand(700, K), _operand(98304, K)
    assert tg._forward_own(700, K, 98304)
    assert tg.supported(x, w) == tg.stats_supported(x, w, 1.0) == tg.gated_supported(x, w) == (K > 0)
    assert _hip_ok(x, _operand(8, 128, K)) == dg.serves(_operand(64, K), _operand(128, K)) == (K > 0)


@pytest.mark.skipif(not L.available(), reason="the kernel library is not built")
def test_entries():
    p, i, n, none = L.c_void_p(1 << 20), L.c_int, L.c_int64, L.c_void_p(0)  # never read
    lib = L.lib()
    assert lib.areal_tgemm_tn(p, n(0), p, n(0), p, n(256), none, i(700), i(256), i(0), i(256), none, i(3), i(1), none) == -1
    assert lib.areal_tgemm_swiglu(p, n(0), p, n(0), p, n(256), i(700), i(256), i(0), i(256), none) == -1
    assert lib.areal_tgemm_grouped(p, p, p, p, p, i(700), i(2), i(256), i(0), n(0), i(0), none) == -1
    assert lib.areal_grouped_gate_up(p, p, p, p, p, i(64), i(2), i(128), i(0), n(0), i(3), none) == -1
    assert lib.areal_grouped_gemm_nt(p, p, p, p, i(64), i(2), i(128), i(0), n(0), i(3), i(0), none) == -1
    assert lib.areal_dgemm(p, n(0), p, none, p, n(128), i(64), i(128), i(0), i(8), i(4), i(0), i(1), i(0), i(0), none) == -1
    assert lib.areal_dswiglu(p, n(0), p, p, n(64), i(64), i(64), i(0), i(4), i(1), i(4), i(0), i(0), none) == -1
