"""Launch plans of row counts that a process has not met: the native search against the Python one, and what a new count costs."""
import random
import time

import pytest

from areal_vllm_amd.ops import attention as A
from areal_vllm_amd.ops import decode_gemm as dg

_rt = pytest.importorskip("areal_vllm_amd._C._runtime")
SHAPES = [(2048, 1536), (1536, 1536), (1536, 8960), (32, 64), (96, 100), (896, 4864), (5120, 13824), (10240, 8192), (28672, 4096), (152064, 3584)]


@pytest.mark.parametrize("N,K", SHAPES)
def test_slab_plan(N, K):
    for M in [*range(1, 130), *range(131, 520, 7), 700, 1000, 2049]:
        assert tuple(_rt.slab_plan(M, N, K)) == dg._slab_plan_py(M, N, K), M


def test_key_ranges():
    r = random.Random(1)
    for _ in range(4000):
        tiles, max_k = int(2 ** r.uniform(0, 13)), int(2 ** r.uniform(0, 18))
        args = tiles, int(tiles * r.uniform(1, 128)), max_k, r.choice([256, 1024]), r.choice([64, 128])
        assert _rt.key_ranges(*args) == A._ranges_py(*args), args


def test_refused():
    for args in [(0, 64, 64), (1, 0, 64), (1, 64, 63)]:
        with pytest.raises(ValueError):
            _rt.slab_plan(*args)
    with pytest.raises(ValueError):
        _rt.key_ranges(0, 1, 1, 1024, 64)


def test_a_new_count_costs_little():
    dg.slab_plan.cache_clear()
    t = time.perf_counter()
    for M in range(1, 513):
        for N, K in SHAPES[:3]:
            dg.slab_plan(M, N, K)
        A.paged_prefill_splits(1, 12, M, 900 + M, M)
    # 8 us; the search in Python takes 280
    assert (time.perf_counter() - t) / 512 < 60e-6
