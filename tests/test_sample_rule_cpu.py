"""How many workgroups the rows of a filtered batch are split over."""
import sys

import pytest

from areal_vllm_amd import ops  # noqa: F401

S = sys.modules["areal_vllm_amd.ops.sampling"]


@pytest.mark.parametrize("V", [100, 8192, 16383, 16384, 32000, 50257, 65536, 151936, 262144])
def test_rounds_and_lengths(V):
    for B in range(1, 385):
        n = S._slices(B, V)
        if V < 2 * S.SLICE_MIN_ENTRIES:
            assert n == 0
            continue
        assert 1 <= n <= 8 and V // n >= S.SLICE_MIN_ENTRIES
        assert B * n <= (512 if B <= 256 else 1024)
