"""Grouped GEMM for expert-sorted tokens (MoE): ``out[t] = x[t] @ W[expert(t)]^T``.

Forward, ``dx`` (on the untransposed weights) and ``dW`` of all experts are one launch each (tiles never straddle experts): the
trainer's 256 x 256 tiles (``csrc/hip/train_gemm.hip``) from 128 rows an expert on, the kernels of ``csrc/hip/grouped_gemm.hip``
below (dW into an fp32 gradient: tiles of 128 x 128 of ``train_gemm.hip``; dW of expert shapes that are no multiples of 128: per
expert with library GEMMs). Counterpart of ``grouped_gemm.ops.gmm`` in the reference
(``realhf/impl/model/modules/moe/experts.py:195-210``).
"""
import itertools
import math
import os
from typing import List, Optional

import torch

from . import _lib as L


def grouped_gemm_ref(x: torch.Tensor, w: torch.Tensor, counts: List[int]) -> torch.Tensor:
    outs, s = [], 0
    for e, n in enumerate(counts):
        if n:
            outs.append(x[s:s + n] @ w[e].t())
        s += n
    return torch.cat(outs, 0) if outs else x.new_zeros(0, w.shape[1])


def _hip_ok(x, w) -> bool:
    return (x.is_cuda and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and w.shape[1] % 64 == 0
            and w.shape[2] % 64 == 0 and w.shape[2] > 0)


# Rows an expert, on average, from which tiles of 256 x 256 (the trainer's dense kernels, operands by LDS-DMA) are the better
# ones although an expert's last row tile is half empty. us of the 64 / 128-row kernels and of these, out / dx / dW:
# 128 experts, 1536 columns, 2048 deep: 64 rows 215 / 198 / 631 and 169 / 177 / 622, 128 321 / 261 / 651 and 225 / 229 / 650,
# 512 669 / 633 / 1037 and 425 / 494 / 862, 1024 1131 / 1123 / 1595 and 729 / 800 / 1163; 2048 columns, 768 deep: 64 99 / 128 /
# 311 and 114 / 111 / 330, 128 134 / 201 / 322 and 134 / 119 / 307, 1024 628 / 746 / 846 and 430 / 389 / 599; 32 experts, 1024 by
# 1024: 64 21 / 22 / 46 and 28 / 29 / 47, 128 28 / 29 / 52 and 29 / 30 / 50.
# They come one a CU: below 54 % of the chip's rounds filled the small ones, of which a CU holds several, are ahead. us small / these,
# out: 4 experts of 400 rows, 2048 columns, 768 deep (33 tiles) 14 / 22; 8 of 128, 4096 columns, 1408 deep (64) 34 / 36; 16 of 400,
# 2048 columns, 768 deep (132 and 264 in all) 21 / 25 and 40 / 44; 16 of 200, 1536 columns (123) 24 / 25; 16 of 400, 2816 columns, 512
# deep (363) 46 / 35.
BIG_MIN_ROWS, BIG_MIN_FILL = 128, 0.54
# dW in fp32, tiles of 256 x 256 / of 128 x 128 (several on a CU, whose products run beside one another's gradients), us: 128 experts of
# 1536 columns, 2048 deep, 128 / 400 / 700 / 1024 / 2048 rows 647 / 548, 840 / 680, 1006 / 863, 1147 / 1076, 1684 / 1833 (the large ones streamed
# past the caches 553, 810, 949, 1092, 1624); 2048 columns, 768 deep 341 / 285, 420 / 349, 492 / 449, 574 / 562, 871 / 991; 8 of 28672 columns, 4096
# deep, 400 / 1024 / 2048 rows 1929 / 1352, 2694 / 2285, 3847 / 4074; 16 of 1536 columns, 768 deep, 1024 rows 69 / 56.
FEW_WGRAD_ROWS = 1024
# Their experts may be large from many rows on only.
BIG_WGRAD_MAX_SIZE, BIG_WGRAD_ANY_SIZE_ROWS = 1 << 24, 2048
# A tile of dW is reduced by one workgroup: behind an expert with many times the mean's rows the chip waits for its few large
# tiles. us of tiles of 128 x 128 (each expert's on all XCDs) / the large ones, largest expert 4 / 8 / 16 / 53 means: 128 experts, 1400
# rows on average, 1536 columns, 2048 deep 1473, 1476, 1483, 1745 and 1412, 1603, 1845, 3032; 2048 columns, 768 deep 874, 878, 930, 1443 and
# 712, 801, 899, 1455; 64 of 2816 columns, 2048 deep 1233, 1266, 1317, 1481 and 1340, 1542, 1939, 3174.
BIG_WGRAD_CROWDED = 8


def _rounds_filled(tiles: float) -> bool:
    return tiles >= BIG_MIN_FILL * 256 * math.ceil(tiles / 256)


def _big_tiles(T: int, E: int, N: int) -> bool:
    """Tiles of 256 x 256 for T rows of E experts and N result columns (half a row tile an expert is empty on average)."""
    return (T >= BIG_MIN_ROWS * E and _rounds_filled((T / 256 + E / 2) * -(-N // 256))
            and "AREAL_GROUPED_GEMM_TILE_M" not in os.environ)


def _big_wgrad(T: int, E: int, N: int, K: int, counts: List[int]) -> bool:
    """Tiles of 256 x 256 for an fp32 dW (not where AREAL_GROUPED_GEMM_TILE_M asks for the small kernels, as for out and dx)."""
    return (T >= FEW_WGRAD_ROWS * E and K % 256 == 0 and (N * K <= BIG_WGRAD_MAX_SIZE or T >= BIG_WGRAD_ANY_SIZE_ROWS * E)
            and _rounds_filled(E * -(-N // 256) * (K // 256)) and max(counts) * E <= BIG_WGRAD_CROWDED * T
            and "AREAL_GROUPED_GEMM_TILE_M" not in os.environ)


def _spread_experts(T: int, E: int, N: int, K: int, counts: List[int]) -> bool:
    """Whether each expert's tiles of 128 x 128 are dealt to all XCDs, not several experts to one. The other XCDs wait for that of a
    crowded expert; its operands pass through eight L2s instead. us dealt by experts / over all, largest expert 1 / 4 / 8 / 16 means:
    128 experts of 500 rows, 1536 columns, 2048 deep (192 tiles) 744 / 725, 786 / 728, 854 / 722, 966 / 729; 2048 columns, 768 deep
    (96) 387 / 424, 410 / 422, 444 / 422, 511 / 424; 8 of 500, 4096 columns, 14336 deep 769 / 796, 1319 / 837, 1756 / 897; 32 of 500,
    1024 by 1024 (64 tiles) 63 / 82, 70 / 83, 89 / 98, 116 / 122; nearly all rows with one expert, 16 of 16 / 64 / 128, 1536 columns, 768 deep
    (72) 14.6 / 10.2, 37.4 / 36.6, 53.0 / 50.1."""
    tiles, most = N // 128 * (K // 128), max(counts)
    return 2 * most > T or tiles >= 80 and most * E > (6 if tiles < 128 else 3 if tiles < 1024 else 1.5) * T


def big_grouped(x: torch.Tensor, w: torch.Tensor, offsets: torch.Tensor, nn: bool) -> torch.Tensor:
    """x[t] @ W[e]^T, or with `nn` x[t] @ W[e], on tiles of 256 x 256 (``csrc/hip/train_gemm.hip``)."""
    T, K = x.shape
    E, N = w.shape[0], w.shape[2 if nn else 1]
    out = torch.empty(T, N, dtype=x.dtype, device=x.device)
    table = torch.empty(4 * (T // 256 + E + 1), dtype=torch.int32, device=x.device)
    L.check(L.lib().areal_tgemm_grouped(L.ptr(x), L.ptr(w), L.ptr(out), L.ptr(offsets), L.ptr(table), L.c_int(T), L.c_int(E),
                                        L.c_int(N), L.c_int(K), L.c_int64(w.stride(0)), L.c_int(int(nn)), L.stream_ptr()),
            "tgemm_grouped")
    return out


def _launch(x: torch.Tensor, w: torch.Tensor, offsets: torch.Tensor) -> torch.Tensor:
    T, K = x.shape
    E, N, K2 = w.shape
    assert K == K2 and offsets.numel() == E + 1 and offsets.dtype == torch.int32 and offsets.is_cuda
    assert x.is_contiguous() and w.stride(2) == 1 and w.stride(1) == K, "operands must be K-contiguous"
    if K % 128 == 0 and w.stride(0) % 8 == 0 and _big_tiles(T, E, N):
        return big_grouped(x, w, offsets, False)
    out = torch.empty(T, N, dtype=x.dtype, device=x.device)
    tile_m = int(os.environ.get("AREAL_GROUPED_GEMM_TILE_M", "0"))  # 0: chosen from the rows per expert
    tm = L.lib().areal_grouped_gemm_tile_m(L.c_int(T), L.c_int(E), L.c_int(N), L.c_int(tile_m))
    L.check(L.lib().areal_grouped_gemm_nt(L.ptr(x), L.ptr(w), L.ptr(out), L.ptr(offsets), L.c_int(T), L.c_int(E),
                                          L.c_int(N), L.c_int(K), L.c_int64(w.stride(0)), L.c_int(T // tm + E),
                                          L.c_int(tile_m), L.stream_ptr()), "grouped_gemm_nt")
    return out


def _fold_target(w: torch.Tensor):
    """The fp32 `main_grad` view of a weight, when its gradient can be accumulated there directly."""
    mg = getattr(w, "main_grad", None)
    return mg if mg is not None and mg.dtype == torch.float32 and mg.is_contiguous() else None


def _after_fold(w: torch.Tensor):
    done = getattr(w, "_after_fold", None)
    if done is not None:  # the gradient went into the fp32 buffer without passing the accumulation hook
        done(w)


class _GroupedGemmFn(torch.autograd.Function):
    """Grouped MFMA kernels: forward, dx on the untransposed weights, dW of all experts in one launch."""

    @staticmethod
    def forward(ctx, x, w, offsets, counts):
        ctx.save_for_backward(x, w, offsets)
        ctx.counts = counts
        return _launch(x, w, offsets)

    @staticmethod
    def backward(ctx, dy):
        x, w, offsets = ctx.saved_tensors
        dy = dy.contiguous()
        dx = dw = None
        E, N, K = w.shape
        if ctx.needs_input_grad[0]:
            if N % 128 == 0 and K % 256 == 0 and _big_tiles(dy.shape[0], E, K) and w.is_contiguous():
                dx = big_grouped(dy, w, offsets, True)
            elif K % 128 == 0:
                # dx[t] = dy[t] @ W[e]: the weights are read as they are (transposed LDS reads in the kernel)
                T = dy.shape[0]
                dx = torch.empty(T, K, dtype=dy.dtype, device=dy.device)
                tile_m = int(os.environ.get("AREAL_GROUPED_GEMM_TILE_M", "0"))
                tm = L.lib().areal_grouped_gemm_tile_m(L.c_int(T), L.c_int(E), L.c_int(K), L.c_int(tile_m))
                L.check(L.lib().areal_grouped_gemm_nn(L.ptr(dy), L.ptr(w), L.ptr(dx), L.ptr(offsets), L.c_int(T),
                                                      L.c_int(E), L.c_int(N), L.c_int(K), L.c_int64(w.stride(0)),
                                                      L.c_int(T // tm + E), L.c_int(tile_m), L.stream_ptr()),
                        "grouped_gemm_nn")
            else:  # the forward kernel on a K-contiguous transposed copy of the weights
                dx = _launch(dy, w.transpose(1, 2).contiguous(), offsets)
        if ctx.needs_input_grad[1]:
            if N % 128 == 0 and K % 128 == 0 and x.shape[0] > 0:
                # dW[e] = dy_e^T . x_e for all experts in one launch (csrc/hip/grouped_gemm.hip); when the weight
                # carries an fp32 `main_grad` view the kernel (csrc/hip/train_gemm.hip) adds into it (no bf16 dW, no separate
                # add kernel)
                mg = _fold_target(w)
                if mg is not None:
                    T = x.shape[0]
                    if _big_wgrad(T, E, N, K, ctx.counts):
                        L.check(L.lib().areal_tgemm_grouped_wgrad(L.ptr(dy), L.ptr(x), L.ptr(mg), L.ptr(offsets), L.c_int(E),
                                                                  L.c_int(N), L.c_int(K), L.c_int64(mg.stride(0)),
                                                                  L.stream_ptr()), "tgemm_grouped_wgrad")
                    else:
                        L.check(L.lib().areal_tgemm_grouped_wgrad_few(
                            L.ptr(dy), L.ptr(x), L.ptr(mg), L.ptr(offsets), L.c_int(max(ctx.counts)), L.c_int(E), L.c_int(N), L.c_int(K),
                            L.c_int64(mg.stride(0)), L.c_int(int(_spread_experts(T, E, N, K, ctx.counts))), L.stream_ptr()), "tgemm_grouped_wgrad_few")
                    _after_fold(w)
                else:
                    dw = torch.empty_like(w)
                    L.check(L.lib().areal_grouped_gemm_wgrad(L.ptr(dy), L.ptr(x), L.ptr(dw), L.ptr(offsets),
                                                             L.c_int(x.shape[0]), L.c_int(E), L.c_int(N), L.c_int(K),
                                                             L.c_int64(dw.stride(0)), L.stream_ptr()), "grouped_gemm_wgrad")
            else:
                dw = torch.zeros_like(w)
                s = 0
                for e, n in enumerate(ctx.counts):
                    if n:
                        torch.mm(dy[s:s + n].t(), x[s:s + n], out=dw[e])
                    s += n
        return dx, dw, None, None


class _LibraryLoopFn(torch.autograd.Function):
    """One library GEMM per expert, forward and backward, written straight into slices of the outputs (no
    concatenation, no per-expert autograd nodes); dW is accumulated by the GEMM into the fp32 `main_grad` view of the
    weight when it has one (``ops/linear.py`` does the same for the dense layers)."""

    @staticmethod
    def forward(ctx, x, w, counts):
        ctx.save_for_backward(x, w)
        ctx.counts = counts
        out = torch.empty(x.shape[0], w.shape[1], dtype=x.dtype, device=x.device)
        s = 0
        for e, n in enumerate(counts):
            if n:
                torch.mm(x[s:s + n], w[e].t(), out=out[s:s + n])
            s += n
        return out

    @staticmethod
    def backward(ctx, dy):
        x, w = ctx.saved_tensors
        dy = dy.contiguous()
        dx = dw = None
        if ctx.needs_input_grad[0]:
            dx = torch.empty_like(x)
            s = 0
            for e, n in enumerate(ctx.counts):
                if n:
                    torch.mm(dy[s:s + n], w[e], out=dx[s:s + n])
                s += n
        if ctx.needs_input_grad[1]:
            mg = _fold_target(w)
            fold = mg is not None and dy.is_cuda and dy.dtype in (torch.bfloat16, torch.float16)
            if not fold:
                dw = torch.zeros_like(w)
            s = 0
            for e, n in enumerate(ctx.counts):
                if n:
                    if fold:
                        torch.addmm(mg[e], dy[s:s + n].t(), x[s:s + n], out_dtype=torch.float32, out=mg[e])
                    else:
                        torch.mm(dy[s:s + n].t(), x[s:s + n], out=dw[e])
                s += n
            if fold:
                _after_fold(w)
        return dx, dw, None


# Few, large experts (Mixtral: 8 experts, thousands of rows each): one library GEMM per expert, at 0.9-1.1 PFLOP/s. The grouped
# kernels are ahead there while the experts' rows are even, and far behind where they are not: a crowded expert's gradient tiles
# are reduced by one workgroup each. us of the library / grouped, forward and backward, 8 experts, 28672 columns, 4096 deep: 1024 rows
# each 7350 / 6259, 2048 10588 / 9385, 1284 to 3000 rows 12061 / 11730, 34 to 9000 rows 12316 / 18765. Many small experts
# (Qwen3-MoE: 128 experts, ~1000 rows each): the loop is launch-bound and the grouped kernel is 2-3x faster
# (tools/grouped_gemm_probe.py). AREAL_GROUPED_GEMM=hip|library overrides the choice.
LIBRARY_MAX_EXPERTS = 16
LIBRARY_MIN_ROWS_PER_EXPERT = 1024


def _prefer_library(n_rows: int, n_experts: int) -> bool:
    forced = os.environ.get("AREAL_GROUPED_GEMM", "auto")
    if forced in ("hip", "library"):
        return forced == "library"
    return n_experts <= LIBRARY_MAX_EXPERTS and n_rows >= LIBRARY_MIN_ROWS_PER_EXPERT * n_experts


def grouped_gemm_offsets_ok(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether `grouped_gemm_offsets` serves these operands."""
    return _hip_ok(x, w) and x.shape[0] > 0


def grouped_gemm_offsets(x: torch.Tensor, w: torch.Tensor, offsets: torch.Tensor) -> torch.Tensor:
    """Forward-only grouped GEMM whose expert row ranges live on the device: x [T, K] rows sorted by expert,
    w [E, N, K], offsets int32 [E + 1] (offsets[e]..offsets[e + 1] = rows of expert e). The launch depends on shapes
    only, so no host synchronisation is needed and the call can be captured into a graph."""
    assert not torch.is_grad_enabled() or not (x.requires_grad or w.requires_grad)
    return _launch(x.contiguous(), w, offsets)


def gate_up_rows_ok(n_pairs: int, w: torch.Tensor) -> bool:
    """Whether `grouped_gate_up` is the kernel for so many rows: its tiles are the small ones, and a column tile holds 64
    gate and 64 up columns."""
    return (0 < n_pairs < BIG_MIN_ROWS * w.shape[0] and "AREAL_GROUPED_GEMM_TILE_M" not in os.environ
            and w.shape[1] % 128 == 0 and w.stride(0) % 8 == 0 and n_pairs // 64 + w.shape[0] <= 65535)


def grouped_gate_up(x: torch.Tensor, src_row: torch.Tensor, w: torch.Tensor, offsets: torch.Tensor) -> torch.Tensor:
    """silu(x[src_row] @ gate^T) * (x[src_row] @ up^T) of every row's expert, forward only, in one launch: x [T, K], src_row
    int64 [R] = the source row of every position of the expert order, w [E, 2 F, K] = gate rows | up rows, offsets int32
    [E + 1] on the device -> [R, F]; the roundings are those of the gather, the grouped GEMM and the activation run apart."""
    x = x.contiguous() if x.data_ptr() % 16 == 0 else x.clone(memory_format=torch.contiguous_format)
    R, K = src_row.numel(), x.shape[1]
    E, N, K2 = w.shape
    assert K == K2 and offsets.numel() == E + 1 and offsets.dtype == torch.int32 and src_row.dtype == torch.int64
    assert w.stride(2) == 1 and w.stride(1) == K and src_row.is_contiguous()
    out = torch.empty(R, N // 2, dtype=x.dtype, device=x.device)
    L.check(L.lib().areal_grouped_gate_up(L.ptr(x), L.ptr(src_row), L.ptr(w), L.ptr(out), L.ptr(offsets), L.c_int(R), L.c_int(E),
                                          L.c_int(N), L.c_int(K), L.c_int64(w.stride(0)), L.c_int(R // 64 + E), L.stream_ptr()),
            "grouped_gate_up")
    return out


def grouped_gemm_rows(x: torch.Tensor, w: torch.Tensor, offsets: torch.Tensor) -> torch.Tensor:
    """Forward-only grouped GEMM for ANY operand shape and for bf16 or fp32 (fp32: true fp32 products): the MFMA
    kernel where it applies, otherwise an LDS-tiled kernel with fp32 accumulation. x [T, K] rows sorted by expert,
    w [E, N, K], offsets int32 [>= E + 1] on the device. No host synchronisation on the GPU."""
    E, N, K = w.shape
    offsets = offsets[:E + 1]
    if x.shape[0] == 0:
        return x.new_zeros(0, N)
    if grouped_gemm_offsets_ok(x, w):
        return _launch(x.contiguous(), w, offsets)
    if L.use_hip(x):
        x = x.contiguous()
        assert w.is_contiguous() and w.dtype == x.dtype and offsets.dtype == torch.int32 and x.shape[1] == K
        out = torch.empty(x.shape[0], N, dtype=x.dtype, device=x.device)
        L.check(L.lib().areal_grouped_gemm_plain(L.ptr(x), L.ptr(w), L.ptr(out), L.ptr(offsets), L.c_int(x.shape[0]),
                                                 L.c_int(E), L.c_int(N), L.c_int(K), L.c_int(L.dtype_flag(x)),
                                                 L.stream_ptr()), "grouped_gemm_plain")
        return out
    off = offsets.tolist()
    return grouped_gemm_ref(x, w, [off[e + 1] - off[e] for e in range(E)])


def grouped_gemm(x: torch.Tensor, w: torch.Tensor, counts: List[int], offsets: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x [T, K] rows sorted by expert, w [E, N, K], counts[e] rows per expert (host ints, sum = T). `offsets`: the same as int32 row
    ranges [E + 1] on x's device, where the caller has them."""
    if _hip_ok(x, w) and x.shape[0] > 0 and _prefer_library(x.shape[0], w.shape[0]):
        L.lib()  # on a GPU box the kernel library must exist even when a shape goes to the GEMM library
        return _LibraryLoopFn.apply(x.contiguous(), w, list(counts))
    if not _hip_ok(x, w) or x.shape[0] == 0:
        if x.is_cuda and x.dtype == torch.bfloat16:
            L.lib()  # on a GPU box the library must exist even when a shape falls back
        return grouped_gemm_ref(x, w, counts)
    if offsets is None:
        offsets = torch.tensor([0] + list(itertools.accumulate(counts)), dtype=torch.int32).to(x.device, non_blocking=True)
    assert offsets.dtype == torch.int32 and offsets.numel() == w.shape[0] + 1
    return _GroupedGemmFn.apply(x.contiguous(), w, offsets, list(counts))
