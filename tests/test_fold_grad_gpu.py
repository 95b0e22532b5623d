"""Addition of small parameters' gradients into the fp32 buffer."""
import pytest
import torch

from areal_vllm_amd import ops

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 8, 1536, 2049, 300001])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_fold_grad(n, dtype):
    g = torch.Generator(device=DEV).manual_seed(n)
    acc = torch.randn(n + 4, device=DEV, generator=g)
    grad = torch.randn(n + 8, device=DEV, generator=g).to(dtype)
    for a, b in ((acc[:n], grad[:n]), (acc[4:], grad[8:]), (acc[1:n], grad[1:n])):  # the last two start unaligned
        want = a + b.float()
        a = a.clone() if a.data_ptr() % 16 == 0 else a
        ops.fold_grad_(a, b)
        assert torch.equal(a, want)
