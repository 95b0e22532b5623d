"""Split-K qkv rows finished by several workgroups a token: blocks of heads that straddle q, k and v, and what is left over."""
import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.ops import decode_gemm as dg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,Hq,Hkv,D,S,norm,fp8", [(1, 1, 1, 16, 1, False, False), (3, 5, 1, 128, 8, True, False),
                                                   (9, 14, 2, 64, 3, False, False), (4, 32, 8, 128, 5, True, True),
                                                   (7, 11, 3, 80, 2, False, False), (2, 3, 2, 256, 4, False, True),
                                                   # many tokens of long rows: a workgroup each; the last ones that are split
                                                   (161, 32, 8, 128, 2, True, False), (240, 64, 8, 128, 1, False, True),
                                                   (160, 32, 8, 128, 2, True, False), (250, 12, 2, 128, 3, False, False)])
def test_heads_dealt_to_blocks(T, Hq, Hkv, D, S, norm, fp8):
    torch.manual_seed(Hq)
    N = (Hq + 2 * Hkv) * D
    cpu = dict(slab=torch.randn(S, T, N), bias=torch.randn(N).bfloat16(), pos=torch.randint(0, 900, (T,), dtype=torch.int32),
               slots=torch.randperm(8 * 32)[:T], qn=torch.rand(D).bfloat16() + 0.5, kn=torch.rand(D).bfloat16() + 0.5)
    cpu["slots"][-1] = -1 if T > 1 else 5  # a padding row: q only
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
    out = []
    for dev in ("cpu", "cuda"):
        a = {k: v.to(dev) for k, v in cpu.items()}
        table = ops.RotaryTable(D, 1024, 1e4, device=dev)
        kc = torch.zeros(8, Hkv, 32, D, device=dev).to(dt)
        vc = torch.zeros(8, Hkv, D, 32, device=dev).to(dt)
        q = dg.splitk_rope_cache_write(a["slab"], S, a["bias"], a["pos"], a["slots"], table, kc, vc, Hq, Hkv, D,
                                       q_norm=a["qn"] if norm else None, k_norm=a["kn"] if norm else None)
        out.append([t.float().cpu() for t in (q, kc, vc)])
    # sums in another order may land on the neighbouring bf16 value (2^-7 of it), and a rotation adds two of them; fp8 steps
    # are 2^-3
    for x, y, step in zip(out[0], out[1], (2.0 ** -7,) + ((2.0 ** -3,) * 2 if fp8 else (2.0 ** -7,) * 2)):
        assert ((x - y).abs() <= 2 * step * x.abs().amax(-1, keepdim=True).clamp(min=1.0)).all()
        assert (x != y).float().mean() < 0.05
