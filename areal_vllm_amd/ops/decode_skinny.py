"""Projections of a decode step of at most 8 rows with the row work around them in the same launch
(``csrc/hip/decode_skinny.hip``). One decoder layer is five launches:

    residual --norm_qkv_rope (RMSNorm, q|k|v, bias, RoPE, KV-cache write)--> q --paged attention-->
    --linear_residual (o)--> residual --norm_gated (RMSNorm, gate|up, activation)--> act --linear_residual (down)--> residual

CPU tensors take PyTorch paths with the same rounding points.
"""
from typing import Optional

import torch
import torch.nn.functional as F

from . import _lib as L
from .decode_gemm import EPI_GEGLU, EPI_SWIGLU, _gate

MAX_ROWS = 8
MAX_NORM_WIDTH = 8192  # values of a normalised row: 8 of them fit the LDS of a CU


def serves(hidden: int, inner: int, q_width: int, head_dim: int) -> bool:
    """Whether the kernels take a layer of this hidden size, MLP width, query width and head size."""
    return (hidden % 64 == 0 and hidden <= MAX_NORM_WIDTH and inner % 64 == 0 and q_width % 64 == 0
            and head_dim % 16 == 0)


def _norm_ref(h, weight, eps, gemma):
    hf = h.float()
    return (hf * torch.rsqrt(hf.pow(2).mean(-1, keepdim=True) + eps)
            * (weight.float() + (1.0 if gemma else 0.0))).to(h.dtype)


def _rows(x: torch.Tensor, w: torch.Tensor) -> None:
    assert x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and x.dim() == 2 and x.shape[0] <= MAX_ROWS
    assert x.stride(1) == 1 and w.is_contiguous() and w.shape[1] == x.shape[1]


def linear_residual(x: torch.Tensor, w: torch.Tensor, residual: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``round(x @ w.T) + residual`` rounded again, bf16 [M, N]."""
    M, K = x.shape
    N = w.shape[0]
    if not L.use_hip(x):
        y = F.linear(x.float(), w.float()).to(x.dtype)
        return y if residual is None else (y.float() + residual.float()).to(x.dtype)
    _rows(x, w)
    assert residual is None or (residual.dtype == x.dtype and residual.shape == (M, N) and residual.is_contiguous())
    y = torch.empty(M, N, dtype=x.dtype, device=x.device)
    L.check(L.lib().areal_skinny_residual(L.ptr(x), L.c_int64(x.stride(0)), L.ptr(w), L.ptr(residual), L.ptr(y), L.c_int(M),
                                          L.c_int(N), L.c_int(K), L.stream_ptr()), "skinny_residual")
    return y


# One row: with two, whose partial results every workgroup would have to combine, the two launches apart are as fast (12 heads of 128 on 2,
# 640 tokens 10.9 / 11.0 us), and the matrix-core form of more rows reads its operand from memory.
PARTS_MAX_WIDTH = 8192  # values of the row, in LDS


def parts_residual(x: torch.Tensor, items, w: torch.Tensor, residual: torch.Tensor) -> torch.Tensor:
    """`linear_residual` of one row of attention output as ``paged_attention_decode(.., items=items, combine=False)`` leaves it: `x`
    or its partial results in `items` (GPU only)."""
    K, N = items.n_q_heads * items.head_dim, w.shape[0]
    assert items.batch == 1 and x.numel() == K <= PARTS_MAX_WIDTH and x.dtype == torch.bfloat16 and x.is_contiguous()
    assert w.dtype == torch.bfloat16 and w.is_contiguous() and w.shape[1] == K
    assert residual.dtype == w.dtype and residual.shape == (1, N) and residual.is_contiguous()
    y = torch.empty(1, N, dtype=w.dtype, device=w.device)
    L.check(L.lib().areal_skinny_parts_residual(L.ptr(x), L.ptr(items.part_o), L.ptr(items.part_ml), L.ptr(items.rows), L.ptr(w),
                                                L.ptr(residual), L.ptr(y), L.c_int(N), L.c_int(items.n_q_heads), L.c_int(items.head_dim),
                                                L.stream_ptr()), "skinny_parts_residual")
    return y


def norm_gated(h: torch.Tensor, norm: torch.Tensor, w_gate_up: torch.Tensor, *, eps: float, gemma: bool = False,
               act: str = "silu") -> torch.Tensor:
    """``act(x @ gate.T) * (x @ up.T)`` of ``x = rmsnorm(h) * norm`` with ``w_gate_up = [gate; up]`` -> bf16 [M, F]."""
    M, K = h.shape
    Fc = w_gate_up.shape[0] // 2
    if not L.use_hip(h):
        y = F.linear(_norm_ref(h, norm, eps, gemma).float(), w_gate_up.float()).to(h.dtype).float()
        return (_gate(y[:, :Fc], EPI_SWIGLU if act == "silu" else EPI_GEGLU) * y[:, Fc:]).to(h.dtype)
    _rows(h, w_gate_up)
    assert norm.dtype == torch.bfloat16 and norm.is_contiguous() and norm.numel() == K
    y = torch.empty(M, Fc, dtype=h.dtype, device=h.device)
    L.check(L.lib().areal_skinny_norm_gated(L.ptr(h), L.c_int64(h.stride(0)), L.ptr(norm), L.ptr(w_gate_up), L.ptr(y),
                                            L.c_int(M), L.c_int(Fc), L.c_int(K), L.c_float(eps), L.c_int(int(gemma)),
                                            L.c_int(0 if act == "silu" else 1), L.stream_ptr()), "skinny_norm_gated")
    return y


def norm_qkv_rope(h: torch.Tensor, norm: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor], positions, slots,
                  table, kcache, vcache, n_q_heads: int, n_kv_heads: int, head_dim: int, *, eps: float,
                  gemma: bool = False, do_rope: bool = True) -> torch.Tensor:
    """The packed q|k|v projection of ``rmsnorm(h) * norm`` with bias; q and k rotated, k and v written into the paged
    caches at ``slots`` (negative: not written); returns the rotated q ``[M, Hq, D]``."""
    M, K = h.shape
    Hq, Hkv, D = n_q_heads, n_kv_heads, head_dim
    if not L.use_hip(h):
        from .attention import rope_and_cache_write_

        y = F.linear(_norm_ref(h, norm, eps, gemma).float(), w.float(), None if bias is None else bias.float())
        qkv = y.to(h.dtype).view(M, Hq + 2 * Hkv, D).contiguous()
        return rope_and_cache_write_(qkv, positions, slots, table, kcache, vcache, Hq, Hkv, do_rope)[:, :Hq].contiguous()
    _rows(h, w)
    assert w.shape[0] == (Hq + 2 * Hkv) * D and norm.dtype == torch.bfloat16 and norm.is_contiguous() and norm.numel() == K
    assert positions.dtype == torch.int32 and slots.dtype == torch.int64 and positions.numel() >= M and slots.numel() >= M
    q = torch.empty(M, Hq, D, dtype=h.dtype, device=h.device)
    L.check(L.lib().areal_skinny_norm_qkv(
        L.ptr(h), L.c_int64(h.stride(0)), L.ptr(norm), L.ptr(w), L.ptr(bias), L.ptr(positions), L.ptr(slots),
        L.ptr(table.cos), L.ptr(table.sin), L.ptr(q), L.ptr(kcache), L.ptr(vcache), L.c_int(M), L.c_int(K), L.c_int(Hq),
        L.c_int(Hkv), L.c_int(D), L.c_int(table.max_pos), L.c_int(int(do_rope)), L.c_float(eps), L.c_int(int(gemma)),
        L.c_int(int(kcache.dtype == torch.float8_e4m3fn)), L.stream_ptr()), "skinny_norm_qkv")
    return q


# One round of the chip's CUs, and as deep as the kernel is ahead of the split-K GEMM and its row kernel (figures at qkv_rows_kernel): with
# 16 rows a workgroup up to 2304 deep (2304 to 4096 columns 9.0 / 8.1 us at 16 rows, 3584 to 4608 12.4 / 16.8), with 32 up to 1536
# (2048 to 2560 columns at 64 rows 10.6 / 15.5); a second round is not (2048 to 3072 columns at 24 rows 8.7 / 10.7).
QKV_ROWS_DEPTH = (2304, 1536)


def qkv_row_tiles(M: int, K: int, N: int, head_dim: int) -> int:
    """16-row tiles of a workgroup of `qkv_rope`, 0 where the split-K GEMM and its row kernel are the faster pair."""
    if K % 64 == 0 and head_dim % 16 == 0:
        for rt in (1, 2):
            if K <= QKV_ROWS_DEPTH[rt - 1] and -(-M // (16 * rt)) * (N // 16) <= 256:
                return rt
    return 0


def qkv_rope(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor], positions, slots, table, kcache, vcache,
             n_q_heads: int, n_kv_heads: int, head_dim: int, row_tiles: int, *, do_rope: bool = True) -> torch.Tensor:
    """The packed q|k|v projection of `x` (normalised rows, any number of them) with bias; q and k rotated, k and v written into
    the paged caches at ``slots`` (negative: not written); returns the rotated q ``[M, Hq, D]``."""
    M, K = x.shape
    Hq, Hkv, D = n_q_heads, n_kv_heads, head_dim
    if not L.use_hip(x):
        from .attention import rope_and_cache_write_

        y = F.linear(x.float(), w.float(), None if bias is None else bias.float())
        qkv = y.to(x.dtype).view(M, Hq + 2 * Hkv, D).contiguous()
        return rope_and_cache_write_(qkv, positions, slots, table, kcache, vcache, Hq, Hkv, do_rope)[:, :Hq].contiguous()
    assert x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and x.stride(1) == 1
    assert w.is_contiguous() and w.shape == ((Hq + 2 * Hkv) * D, K) and (bias is None or bias.dtype == torch.bfloat16 and bias.is_contiguous())
    assert positions.dtype == torch.int32 and slots.dtype == torch.int64 and positions.numel() >= M and slots.numel() >= M
    q = torch.empty(M, Hq, D, dtype=x.dtype, device=x.device)
    L.check(L.lib().areal_qkv_rows(
        L.ptr(x), L.c_int64(x.stride(0)), L.ptr(w), L.ptr(bias), L.ptr(positions), L.ptr(slots), L.ptr(table.cos), L.ptr(table.sin),
        L.ptr(q), L.ptr(kcache), L.ptr(vcache), L.c_int(M), L.c_int(K), L.c_int(Hq), L.c_int(Hkv), L.c_int(D), L.c_int(table.max_pos),
        L.c_int(int(do_rope)), L.c_int(int(kcache.dtype == torch.float8_e4m3fn)), L.c_int(row_tiles), L.stream_ptr()), "qkv_rows")
    return q
