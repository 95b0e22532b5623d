"""Which prefills run on the decode step's GEMMs: by rows, hidden size and what the row kernels take."""
from types import SimpleNamespace

import pytest
import torch

from areal_vllm_amd.inference.model_runner import ModelRunner


@pytest.mark.parametrize("rows,hidden,heads,taken", [
    (0, 1536, (12, 2, 128, False), False), (1, 1536, (12, 2, 128, False), True), (512, 4096, (32, 8, 128, False), True),
    (513, 1536, (12, 2, 128, False), False), (256, 8192, (64, 8, 128, False), True), (257, 8192, (64, 8, 128, False), False),
    (257, 5120, (40, 8, 128, False), False), (64, 1024, (120, 8, 128, False), False), (64, 1024, (112, 8, 128, False), True),
    (64, 1024, (8, 8, 96, True), False), (64, 1024, (8, 8, 96, False), True), (64, 1024, (8, 8, 64, True), True)])
def test_rule(rows, hidden, heads, taken):
    hq, hkv, D, qk_norm = heads
    r = SimpleNamespace(cfg=SimpleNamespace(head_dim=D, hidden_size=hidden, qk_norm=qk_norm), hq=hq, hkv=hkv, fused_decode=True,
                        dtype=torch.bfloat16, PREFILL_FUSED_MAX_ROWS=ModelRunner.PREFILL_FUSED_MAX_ROWS,
                        PREFILL_FUSED_MAX_ROWS_WIDE=ModelRunner.PREFILL_FUSED_MAX_ROWS_WIDE)
    assert ModelRunner._prefill_fused(r, rows) == taken
