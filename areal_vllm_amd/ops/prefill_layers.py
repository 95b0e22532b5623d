"""All layers of a short prefill behind cached context, queued by one native call (``csrc/hip/prefill_layers.hip``): the launches
that ``ModelRunner._prefill_layers_fused`` makes one by one, on the same kernels and plans and with the same results.

Role in the reference: the serving engine's prefill step (areal/api/cli_args.py:398-454)."""
import ctypes
import itertools
from typing import Optional

import numpy as np
import torch

from . import _lib as L
from . import decode_gemm as dg
from .attention import PAGE_SIZE, is_fp8, paged_prefill_splits

P, I = ctypes.c_void_p, ctypes.c_int


class _Pass(ctypes.Structure):
    _fields_ = ([(n, P) for n in ("layers", "first", "x", "stream", "res0", "res1", "slab", "q", "attn", "act", "part", "pos", "slots", "cos", "sin",
                                  "block_tables", "cu_q", "cu_k")]
                + [(n, I) for n in ("n_layers", "T", "H", "F", "Hq", "Hkv", "D", "max_pos", "max_pages", "B", "max_q", "splits")]
                + [(n, I * 3) for n in ("qkv_plan", "o_plan", "down_plan")]
                + [(n, I) for n in ("gate_cols", "gate_blocks", "act_kind", "fp8", "gemma")]
                + [("eps", ctypes.c_float), ("scale", ctypes.c_float)])


def _aligned(t: Optional[torch.Tensor], dtype: torch.dtype) -> bool:
    return t is None or (t.is_cuda and t.dtype == dtype and t.is_contiguous() and t.data_ptr() % 16 == 0)


# Layers of the first native calls; the last one takes the others. Naming a layer's tensors to the kernels is 8 us on the host, a layer 60 to
# 80 on the device: it starts behind the first two and never waits for the rest. 93 tokens, 28 layers, behind 811: named all at once the
# first launch of a layer came 310 us after its inputs, of 2410 in all; 90 of 2140 now.
LEADING = (2, 6)


def _addresses(layers, kv, shapes, cache) -> Optional[np.ndarray]:
    """The layers' addresses as the kernels take them, None where an operand is not for them."""
    bf, out = torch.bfloat16, []
    for ws, caches in zip(layers, kv):
        for w, s in zip(ws, shapes):
            if w is None:
                out.append(0)
            elif w.shape == s and w.dtype is bf and w.is_cuda and w.is_contiguous():
                out.append(w.data_ptr())
            else:
                return None
        if (ws[2] is None) != (ws[3] is None):
            return None
        for c in caches:
            if not (c.dtype is cache and c.is_cuda and c.is_contiguous()):
                return None
            out.append(c.data_ptr())
    out = np.array(out, dtype=np.uint64)
    return out if int(np.bitwise_or.reduce(out)) % 16 == 0 else None


def run(layers, kv, x, residual, positions, slots, rope, cu_q, cu_k, block_tables, max_q: int, n_q_heads: int, n_kv_heads: int,
        head_dim: int, eps: float, gemma: bool, act: str) -> Optional[torch.Tensor]:
    """layers: per layer (qkv, qkv bias or None, q norm or None, k norm or None, o, second norm, gate_up, down, norm behind the
    layer or None for the last), asked for as they are needed; kv: the layers' caches; x, residual [T, H]: the first layer's
    normalised input and the residual stream (both kept). Returns the residual stream behind the last layer, or None where these
    operands are for the single launches (another type, layout or head size; layers ahead of the first that is have run then, to no
    effect but that they have written their keys and values)."""
    T, H = x.shape
    Hq, Hkv, D = n_q_heads, n_kv_heads, head_dim
    N, HD = (Hq + 2 * Hkv) * D, Hq * D
    bf, i32 = torch.bfloat16, torch.int32
    layers = iter(layers)
    ahead = list(itertools.islice(layers, LEADING[0]))
    F = ahead[0][7].shape[1]
    gate = dg.swiglu_plan(T, F)
    if not (x.is_cuda and 0 < T <= dg.MAX_ROWS and D == 128 and gate is not None and H % 64 == 0 and F % 64 == 0
            and _aligned(x, bf) and _aligned(residual, bf) and _aligned(block_tables, i32) and block_tables.dim() == 2
            and positions.dtype == i32 and slots.dtype == torch.int64 and cu_q.dtype == i32 and cu_k.dtype == i32
            and positions.is_contiguous() and slots.is_contiguous() and positions.numel() == T and slots.numel() == T):
        return None
    fp8 = is_fp8(kv[0][0])
    cache = torch.float8_e4m3fn if fp8 else bf
    shapes = ((N, H), (N,), (D,), (D,), (H, HD), (H,), (2 * F, H), (H, F), (H,))
    table = _addresses(ahead, kv, shapes, cache)
    if table is None:
        return None
    plans = [dg.slab_plan(T, n, k) for n, k in ((N, H), (H, HD), (H, F))]
    B = cu_q.numel() - 1
    splits = paged_prefill_splits(B, Hq, max_q, block_tables.shape[1] * PAGE_SIZE, T)
    dev = x.device
    new = lambda *shape, dtype=bf: torch.empty(*shape, dtype=dtype, device=dev)
    between, res, normed = new(T, H), new(T, H), new(T, H)
    slab = new(max(p[2] * n for p, n in zip(plans, (N, H, H))) * T, dtype=torch.float32)
    q, attn, acts = new(T, HD), new(T, HD), new(T, F)
    part = new(splits * T * Hq * (D + 2), dtype=torch.float32) if splits > 1 else None
    a = _Pass(T=T, H=H, F=F, Hq=Hq, Hkv=Hkv, D=D, max_pos=rope.max_pos, max_pages=block_tables.shape[1], B=B, max_q=max_q, splits=splits,
              gate_cols=gate[0], gate_blocks=gate[1], act_kind=0 if act == "silu" else 1, fp8=int(fp8), gemma=int(bool(gemma)),
              eps=float(eps), scale=D ** -0.5)
    for name, t in (("first", x), ("x", normed), ("stream", residual), ("res0", between), ("res1", res), ("slab", slab), ("q", q), ("attn", attn), ("act", acts),
                    ("part", part), ("pos", positions), ("slots", slots), ("cos", rope.cos), ("sin", rope.sin),
                    ("block_tables", block_tables), ("cu_q", cu_q), ("cu_k", cu_k)):
        setattr(a, name, None if t is None else t.data_ptr())
    for name, p in zip(("qkv_plan", "o_plan", "down_plan"), plans):
        setattr(a, name, (I * 3)(*p))
    done = 0
    for size in (*LEADING[1:], None):
        a.layers, a.n_layers = table.ctypes.data, len(ahead)
        L.check(L.lib().areal_prefill_layers(ctypes.byref(a), L.stream_ptr()), "prefill_layers")
        done += len(ahead)
        a.first, a.stream = a.x, a.res1
        ahead = list(itertools.islice(layers, size))
        if not ahead:
            return res
        table = _addresses(ahead, kv[done:], shapes, cache)
        if table is None:
            return None
    a.layers, a.n_layers = table.ctypes.data, len(ahead)
    L.check(L.lib().areal_prefill_layers(ctypes.byref(a), L.stream_ptr()), "prefill_layers")
    return res
