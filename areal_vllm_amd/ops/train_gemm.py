"""Hand-written dense bf16 GEMM for the trainer and for prefill (``csrc/hip/train_gemm.hip``).

``tgemm_tn(a, b)`` = ``a @ b.T`` for K-contiguous operands (activations x ``nn.Linear`` weight), ``tgemm_nn(dy, w)`` =
``dy @ w`` on the weight as it lies in memory (input gradient), ``tgemm_wgrad_`` adds ``dy.T @ x`` to an fp32 gradient,
``logit_stats`` reduces a vocabulary's logits without writing them. The kernels cover the shapes transformer layers produce (K a
multiple of 128, N of 4, 16-byte aligned rows); `supported()` and the rules beside `forward` and `dgrad` tell the caller when to
keep the library GEMM instead - statements about shapes, not a fallback for a missing extension (on a GPU the extension is
mandatory)."""
import functools
import os
from typing import Optional, Tuple

import torch
from torch.autograd import forward_ad

from . import _lib as L

# AREAL_OWN_WGRAD=0 sends weight gradients back to the library GEMM (A/B runs on one box)
OWN_WGRAD = os.environ.get("AREAL_OWN_WGRAD", "1") != "0"


def supported(a: torch.Tensor, b: torch.Tensor, bias: Optional[torch.Tensor] = None) -> bool:
    if not (a.is_cuda and a.dtype == torch.bfloat16 and b.dtype == torch.bfloat16 and a.dim() == 2 and b.dim() == 2):
        return False
    M, K = a.shape
    N = b.shape[0]
    if b.shape[1] != K or K % 128 != 0 or K == 0 or N % 4 != 0 or M == 0:
        return False
    if a.stride(1) != 1 or b.stride(1) != 1 or a.stride(0) % 8 or b.stride(0) % 8:
        return False
    if a.data_ptr() % 16 or b.data_ptr() % 16:
        return False
    if bias is not None and (bias.dtype != torch.bfloat16 or not bias.is_contiguous() or bias.data_ptr() % 8):
        return False
    return True


def tgemm_tn(a: torch.Tensor, b: torch.Tensor, bias: Optional[torch.Tensor] = None,
             out: Optional[torch.Tensor] = None, max_blocks: int = 256, plan: Optional[Tuple[int, int]] = None) -> torch.Tensor:
    """out[M, N] = a[M, K] @ b[N, K]^T (+ bias[N]); bf16 in, fp32 accumulation, bf16 out. `plan`: (tiles reduced by one
    workgroup, parts of the others) of ``_tile_plan``, without a bias."""
    M, K = a.shape
    N = b.shape[0]
    if out is None:
        out = torch.empty(M, N, dtype=torch.bfloat16, device=a.device)
    assert supported(a, b, bias) and out.dtype == torch.bfloat16 and out.stride(1) == 1 and out.stride(0) % 4 == 0
    whole, splits = plan or (0, 1)
    part = None
    if splits > 1:
        part = torch.empty(splits * (-(-M // 256) * -(-N // 256) - whole) << 16, dtype=torch.float32, device=a.device)
    L.check(L.lib().areal_tgemm_tn(L.ptr(a), L.c_int64(a.stride(0)), L.ptr(b), L.c_int64(b.stride(0)), L.ptr(out),
                                   L.c_int64(out.stride(0)), L.ptr(bias), L.c_int(M), L.c_int(N), L.c_int(K),
                                   L.c_int(int(max_blocks)), L.ptr(part), L.c_int(whole), L.c_int(splits), L.stream_ptr()),
            "tgemm_tn")
    return out


MAX_ROW_STRIDE = 1 << 24  # elements: byte offsets inside 64 rows of an operand fit 32 bits


def wgrad_supported(dy: torch.Tensor, x: torch.Tensor, acc: torch.Tensor) -> bool:
    if not OWN_WGRAD:
        return False
    if not (dy.is_cuda and dy.dtype == torch.bfloat16 and x.dtype == torch.bfloat16 and acc.dtype == torch.float32):
        return False
    if dy.dim() != 2 or x.dim() != 2 or dy.shape[0] != x.shape[0] or acc.shape != (dy.shape[1], x.shape[1]):
        return False
    M, N = dy.shape
    K = x.shape[1]
    if N % 128 or K % 256 or M < 256:
        return False
    if dy.stride(1) != 1 or x.stride(1) != 1 or acc.stride(1) != 1 or dy.stride(0) % 8 or x.stride(0) % 8:
        return False
    if dy.stride(0) < N or x.stride(0) < K:  # repeated or overlapping rows: the end of the operand is told from a row's place
        return False
    if dy.stride(0) > MAX_ROW_STRIDE or x.stride(0) > MAX_ROW_STRIDE:
        return False
    return dy.data_ptr() % 16 == 0 and x.data_ptr() % 16 == 0


def _even_splits(pairs: int, splits: int) -> int:
    """At most `splits` parts of `pairs`, none of them empty."""
    splits = max(1, min(splits, pairs))
    return -(-pairs // -(-pairs // splits))


@functools.lru_cache(maxsize=1024)
def _tile_plan(pairs: int, tiles: int, flush: int, rows: int = 256) -> Tuple[float, int, int]:
    """(time in 128-deep pairs, 3 us each; tiles of 256 x 256 that one workgroup reduces; parts of the reduction of each of the
    others). A CU runs one workgroup: tiles beyond a multiple of 256 would leave CUs idle in a last round, so they are split
    until the round is full. `flush`: pairs that writing a whole tile's result takes. A part costs 6 pairs more (its start, and
    256 KiB of fp32 to write; half of it for the few `rows` of a single row tile), a chip full of them 8 to be read and summed, the
    summing kernel itself 2 and a 24th for each part that a thread adds: 48 tiles of 256 pairs in
    5 parts take 183 us, 210 tiles in 6 parts (330 MB, more than the memory-side cache holds) 871, whole 745 (the 46 CUs that
    idle leave their power to the others)."""
    rounds, rest = divmod(tiles, 256)
    best = (float(-(-tiles // 256) * (pairs + flush)), tiles, 1)
    if rest:
        for s in range(2, min(pairs, 64) + 1):
            chunk = -(-pairs // s)
            if -(-pairs // chunk) == s:  # (every part has work)
                cost = (rounds * (pairs + flush) + -(-rest * s // 256) * (chunk + 3 + 3 * rows / 256) + 2
                        + 8 * s * rest / 256 * rows / 256 + s / 24)
                best = min(best, (cost, rounds * 256, s))
    return best


def _wgrad_few(M: int, tiles: int) -> bool:
    """Whether `tiles` of 128 x 128, several on a CU, are the better ones over M tokens where the large ones are not split; us of the
    tiles of 256 x 256 / of these, the gradient not in the caches. Up to three tiles a CU 2 tiles, 600 tokens 10.5 / 9.6; 16 tiles, 600
    13.5 / 10; 768, 256 / 700 / 1280 / 3072 29.5 / 23.2, 37.6 / 30.3, 47.3 / 40.9, 78 / 76. Not where they fill most of one round, for
    what they lose with the gradient in the memory-side cache is more than they gain without: 780 tiles, 256 / 700 / 1024 29.6 / 26.5,
    38.7 / 37.1, 43.5 / 44.9 and 23.6 / 25.7, 32.9 / 38.5, 37.9 / 45.7; 840 29.9 / 27.1, 39.3 / 37.6, 45.5 / 45.3 and 25.0 / 26.0, 34.5 /
    38.3, 39.4 / 45.9; 900 31.1 / 27.9, 41.0 / 38.6, 47.0 / 46.3 and 26.0 / 27.2, 36.0 / 39.6, 41.2 / 47.2; from 960 on 33.2 / 27.2, 43.5 /
    37.7, 49.0 / 46.2 and 28.3 / 27.1, 38.7 / 38.6, 44.0 / 46.7. More: 1200, 1500 88 / 73; 1680, 700 / 1500 / 2048 78 / 61, 107 / 93, 127 /
    117; 5504, 1024 / 1500 / 2048 270 / 211, 330 / 293, 394 / 392; but full rounds, 1008, 1024 / 1500 51 / 47, 61 / 59; 14244, 1024 / 1500
    637 / 599, 789 / 798."""
    if tiles <= 768:
        return M <= min(3072, 600 + 11 * tiles)
    filled = tiles / 1024 / -(-tiles // 1024)
    return tiles >= 960 and M <= (1536 if filled <= 0.92 else 1024)


def tgemm_wgrad_(acc: torch.Tensor, dy: torch.Tensor, x: torch.Tensor, splits: int = 0) -> torch.Tensor:
    """acc[N, K] (fp32) += dy[M, N]^T @ x[M, K]: the weight gradient of ``y = x @ W^T`` summed straight into the
    fp32 gradient buffer. `splits`: parts of the token range for every tile (0: chosen)."""
    assert wgrad_supported(dy, x, acc)
    (M, N), K = dy.shape, x.shape[1]
    pairs, tiles = -(-M // 128), -(-N // 256) * (K // 256)
    if splits:
        splits = _even_splits(pairs, splits)
        whole = 0 if splits > 1 else tiles
    else:
        # (reading, adding to and writing a tile's gradient: 1500 tokens, 1536 x 1536, 36 tiles whole / in 3 parts 37 / 28 us, 48
        # tiles 38 / 31, 100 tiles 40 / 58)
        _, whole, splits = _tile_plan(pairs, tiles, 5)
        # Parts sum in shorter chains: in place of whole tiles only the small ones give the same bits. Relative error against 64 bits in
        # parts / in one chain, 512 x 512, 700 tokens 7.7e-8 / 1.5e-7, 2048 x 1536, 1500 1.3e-7 / 2.3e-7 (31 / 22 us).
        if splits == 1 and _wgrad_few(M, N // 128 * (K // 128)):
            L.check(L.lib().areal_tgemm_wgrad_few(L.ptr(dy), L.c_int64(dy.stride(0)), L.ptr(x), L.c_int64(x.stride(0)), L.ptr(acc),
                                                  L.c_int64(acc.stride(0)), L.c_int(M), L.c_int(N), L.c_int(K), L.stream_ptr()),
                    "tgemm_wgrad_few")
            return acc
    part = torch.empty(splits * (tiles - whole) << 16, dtype=torch.float32, device=dy.device) if splits > 1 else None
    L.check(L.lib().areal_tgemm_wgrad(L.ptr(dy), L.c_int64(dy.stride(0)), L.ptr(x), L.c_int64(x.stride(0)), L.ptr(acc),
                                      L.c_int64(acc.stride(0)), L.c_int(M), L.c_int(N), L.c_int(K), L.c_int(splits),
                                      L.c_int(whole), L.ptr(part), L.stream_ptr()), "tgemm_wgrad")
    return acc


def dgrad_cost(M: int, R: int, C: int) -> Tuple[float, int, int]:
    return _tile_plan(R // 128, -(-M // 256) * (C // 256), 0, min(256, -(-M // 32) * 32))


def dgrad_supported(dy: torch.Tensor, w: torch.Tensor) -> bool:
    if not (dy.is_cuda and dy.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and dy.dim() == 2 and w.dim() == 2):
        return False
    M, R = dy.shape
    if w.shape[0] != R or M == 0 or R == 0 or R % 128 or w.shape[1] % 256 or w.shape[1] == 0:
        return False
    if dy.stride(1) != 1 or w.stride(1) != 1 or dy.stride(0) % 8 or w.stride(0) % 8:
        return False
    if not (R <= dy.stride(0) <= 1 << 22 and w.shape[1] <= w.stride(0) <= MAX_ROW_STRIDE):  # (256 rows of dy)
        return False
    return dy.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0


def tgemm_nn(dy: torch.Tensor, w: torch.Tensor, splits: int = 0, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """dy[M, R] @ w[R, C] in bf16 with fp32 accumulation: the input gradient of ``y = x @ W^T`` from the weight as it lies."""
    assert dgrad_supported(dy, w)
    (M, R), C = dy.shape, w.shape[1]
    tiles = -(-M // 256) * (C // 256)
    whole, splits = (0 if splits > 1 else tiles, splits) if splits else dgrad_cost(M, R, C)[1:]
    if out is None:
        out = torch.empty(M, C, dtype=torch.bfloat16, device=dy.device)
    assert out.shape == (M, C) and out.dtype == torch.bfloat16 and out.is_contiguous()
    part = torch.empty(splits * (tiles - whole) << 16, dtype=torch.float32, device=dy.device) if splits > 1 else None
    L.check(L.lib().areal_tgemm_nn(L.ptr(dy), L.c_int64(dy.stride(0)), L.ptr(w), L.c_int64(w.stride(0)), L.ptr(out),
                                   L.c_int64(C), L.ptr(part), L.c_int(whole), L.c_int(splits), L.c_int(M), L.c_int(R),
                                   L.c_int(C), L.stream_ptr()), "tgemm_nn")
    return out


# Own kernel / library, us (the weight as it lies; the library is 8 to 20 % slower in this layout than with a transposed copy).
# Deep reductions, at any row count: 17920 deep to 1536 columns, 256 / 700 / 3000 / 12000 / 32768 rows 38 / 109, 55 / 133,
# 173 / 222, 488 / 912, 1281 / 1324; 151936 to 1536, 256 / 700 / 6000 rows 144 / 466, 281 / 607, 2195 / 4089; 37888 to 3584,
# 700 / 32768 rows 172 / 341, 6169 / 6466. Short ones: 1536 deep to 8960 columns, 700 / 1500 / 12000 / 32768 rows 38 / 33,
# 41 / 49, 257 / 290, 682 / 755; 2048 to 4096, 1500 / 3000 / 32768 rows 46 / 33, 48 / 49, 386 / 439; 2048 to 1536, 700 / 6000 /
# 12000 / 32768 rows 31 / 22, 46 / 42, 78 / 100, 148 / 161. So: a deep reduction, or rounds that are
# filled to five eighths (384 tiles 16 pairs deep: 92 / 90; 288 tiles 8 deep, two rounds for 1.1: 53 / 49; 1536 deep to 1536, 144 tiles: 35 / 33).
# A deep reduction of one round of tiles that splitting does not fill is the library's: 10000 rows, 8192 deep to 1024 columns (160
# tiles) 142 / 136, 3000 rows, 28672 deep to 4096 (192) 590 / 560; filled, it is not: 37888 deep to 3584 (168) 636 / 1057.
DGRAD_MIN_DEPTH, DGRAD_MIN_TILES, DGRAD_MAX_LOSS, DGRAD_MAX_ROUND_LOSS = 8192, 192, 1.6, 1.25


@functools.lru_cache(maxsize=1024)
def _dgrad_own(M: int, R: int, C: int) -> bool:
    tiles = -(-M // 256) * (C // 256)
    if R >= DGRAD_MIN_DEPTH:
        return not 128 < tiles < 256 or dgrad_cost(M, R, C)[0] <= DGRAD_MAX_ROUND_LOSS * tiles * (R // 128) / 256
    return tiles >= DGRAD_MIN_TILES and dgrad_cost(M, R, C)[0] <= DGRAD_MAX_LOSS * M * (C // 256) * (R // 128) / 65536


def dgrad(dy: torch.Tensor, w: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """dy @ w inside a backward pass (a library product where that pass is itself recorded)."""
    if (not torch.is_grad_enabled() and dgrad_supported(dy, w) and (out is None or out.is_contiguous() and out.data_ptr() % 8 == 0
                                                                    and out.dtype == torch.bfloat16)):
        if _dgrad_own(dy.shape[0], *w.shape):
            return tgemm_nn(dy, w, out=out)
    return torch.mm(dy, w) if out is None else torch.mm(dy, w, out=out)


# Where the own kernel is ahead of the library in y = x W^T, own / library us (the library's choices jump: of 70 depths and widths
# those below are where the own one is ahead or level: 0.69 of its time in the mean of 273 sizes, 12 of them 3 to 16 % behind).
# Deep reductions of up to 128 tiles, which it splits: 8960 deep to 1536 columns, 800 / 1500 / 2048 rows 40 / 46, 52 / 69, 61 / 70;
# 11008 to 4096, 1100 rows 99 / 121; 18944 to 3584, 257 / 800 rows 66 / 93, 120 / 164. A few tiles of 9 to 16 thousand deep are the
# library's (8960 to 512, 800 rows 29 / 25), so are 8192 deep ones (1536 columns, 800 rows 38 / 35) and 96 and more tiles of 8192
# columns (11008 deep, 600 rows 134 / 126). More tiles: rounds that are not full, from 16384 deep on: 18944 to 4096, 4500 rows (288
# tiles) 0.49 of the library's time, to 5120, 9000 rows (720) 0.76; but to 3584, 9000 rows (504) 867 / 822, and one round of more
# than 128 (160 to 256 tiles) 4 to 19 % slower.
# Wide results, stored by whole lines: 1536 deep to 151936 columns, 300 / 700 / 1500 / 3000 / 8192 rows 192 / 187, 285 / 354, 578 /
# 639, 1154 / 1171, 2890 / 2984; 128256 columns, 896 / 5120 deep, 1642 rows 0.91 / 0.94 of the library's time, but 3584 and 4096 deep
# 2500 to 8192 rows 1.01 to 1.06 of it, and 65536 columns from 2500 rows on 1.02 to 1.13.
def _forward_own(M: int, K: int, N: int) -> bool:
    if N >= 98304:
        return M >= 600 and (K <= 3072 or K >= 4608)
    if K < 8704 or not 256 < M <= 12288 or N >= 65536:
        return False
    tiles = -(-M // 256) * -(-N // 256)
    if tiles <= 128:
        return K >= 16384 or 600 <= M <= 2048 and N <= 6144 and tiles * K >= 150000
    return K >= 16384 and 256 < tiles <= 0.95 * 256 * -(-tiles // 256)


# Logits that are reduced, not written, us of that form / of the library's product and the pass over its logits: 151936 columns, 896
# to 5120 deep, 600 to 8192 rows 0.75 to 1.02 of its time, 65536 columns, 896 / 2048 deep 0.87 to 0.98 / 0.95 to 1.04; 3584 and 4096
# deep 1.00 to 1.12, with 100352 columns 0.90 to 1.08; 151936 of them 4096 deep, 4000 / 8192 / 13019 rows 1.00 / 1.02 / 1.04.
def _stats_own(M: int, K: int, N: int) -> bool:
    return N >= 65536 and M >= 600 and (K <= 3072 or N >= 98304 and (M <= 4096 or K <= 3584 or K >= 4608))


def plain(*tensors: torch.Tensor) -> bool:
    """Whether a kernel on raw pointers may stand in for an ATen product of these tensors: nothing rewrites or records the call
    (vmap and its like, tracing and compilation, dispatch and function modes, autocast), and no operand is a subclass or a dual."""
    return not (torch._C._are_functorch_transforms_active() or torch._C._len_torch_dispatch_stack()
                or torch._C._len_torch_function_stack() or torch.jit.is_tracing() or torch.compiler.is_compiling()
                or torch.is_autocast_enabled(tensors[0].device.type)
                or any(type(t) not in (torch.Tensor, torch.nn.Parameter) or forward_ad.unpack_dual(t).tangent is not None
                       for t in tensors))


def forward(x: torch.Tensor, w: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x[M, K] @ w[N, K]^T outside autograd."""
    if (x.dim() == 2 and w.dim() == 2 and _forward_own(x.shape[0], w.shape[1], w.shape[0]) and plain(x, w) and supported(x, w)
            and w.shape[0] % 8 == 0 and (out is None or out.dtype == torch.bfloat16 and out.stride(1) == 1
                                         and out.stride(0) % 8 == 0 and out.data_ptr() % 16 == 0)):
        _, whole, splits = _tile_plan(x.shape[1] // 128, -(-x.shape[0] // 256) * -(-w.shape[0] // 256), 0)
        return tgemm_tn(x, w, out=out, plan=(whole, splits))
    return torch.mm(x, w.t(), out=out) if out is not None else torch.nn.functional.linear(x, w)


def stats_supported(x: torch.Tensor, w: torch.Tensor, temperature: float) -> bool:
    """Whether `logit_stats` is the kernel for these logits."""
    return (0.0 < temperature < float("inf") and x.dim() == 2 and w.dim() == 2
            and _stats_own(x.shape[0], w.shape[1], w.shape[0]) and supported(x, w))


def logit_stats(x: torch.Tensor, w: torch.Tensor, labels: torch.Tensor, temperature: float, vocab_start: int,
                out: torch.Tensor) -> None:
    """out[4, M] (rows with unit stride) = ``ops.logprob.logprob_stats`` of the logits x[M, K] @ w[N, K]^T (in bf16), which are
    not written."""
    M, K = x.shape
    N = w.shape[0]
    assert labels.dtype == torch.int64 and labels.is_contiguous() and labels.numel() == M
    assert out.dtype == torch.float32 and out.shape == (4, M) and out.stride(1) == 1
    part = torch.empty(3 * ((N + 63) // 64) * M, dtype=torch.float32, device=x.device)
    L.check(L.lib().areal_tgemm_stats(L.ptr(x), L.c_int64(x.stride(0)), L.ptr(w), L.c_int64(w.stride(0)), L.ptr(labels),
                                      L.c_int64(vocab_start), L.c_int(M), L.c_int(N), L.c_int(K), L.c_float(1.0 / temperature),
                                      L.ptr(part), L.ptr(out[0]), L.ptr(out[1]), L.ptr(out[2]), L.ptr(out[3]), L.stream_ptr()),
            "tgemm_stats")


# rows from which the fused gate|up + SwiGLU kernel replaces library GEMM + activation kernel in no-grad forwards
GATED_MIN_ROWS = int(os.environ.get("AREAL_FUSED_MLP_MIN_ROWS", "4096"))


def gated_supported(x: torch.Tensor, w_gate_up: torch.Tensor) -> bool:
    if not (x.is_cuda and x.dim() == 2 and w_gate_up.dim() == 2 and x.dtype == torch.bfloat16
            and w_gate_up.dtype == torch.bfloat16):
        return False
    M, K = x.shape
    if w_gate_up.shape[1] != K or w_gate_up.shape[0] % 2 or K % 128 or K == 0 or (w_gate_up.shape[0] // 2) % 4:
        return False
    if x.stride(1) != 1 or x.stride(0) % 8 or not w_gate_up.is_contiguous():
        return False
    return x.data_ptr() % 16 == 0 and w_gate_up.data_ptr() % 16 == 0 and M > 0


def tgemm_swiglu(x: torch.Tensor, w_gate_up: torch.Tensor, out: Optional[torch.Tensor] = None,
                 max_blocks: int = 256) -> torch.Tensor:
    """out[M, F] = silu(x @ Wg^T) * (x @ Wu^T) for W = [Wg; Wu] of shape [2 F, K]: the gate|up projection of a gated
    MLP and its activation in one kernel (gate and up are rounded to bf16 before the activation, as the unfused path
    holds them); the [M, 2 F] intermediate is never written. For forward passes that keep no activations."""
    assert gated_supported(x, w_gate_up)
    M, K = x.shape
    Fo = w_gate_up.shape[0] // 2
    if out is None:
        out = torch.empty(M, Fo, dtype=torch.bfloat16, device=x.device)
    assert out.dtype == torch.bfloat16 and out.stride(1) == 1 and out.stride(0) % 4 == 0
    L.check(L.lib().areal_tgemm_swiglu(L.ptr(x), L.c_int64(x.stride(0)), L.ptr(w_gate_up), L.c_int64(w_gate_up.stride(0)),
                                       L.ptr(out), L.c_int64(out.stride(0)), L.c_int(M), L.c_int(Fo), L.c_int(K),
                                       L.c_int(int(max_blocks)), L.stream_ptr()), "tgemm_swiglu")
    return out


def gate_up_act(x: torch.Tensor, w_gate_up: torch.Tensor, act: str = "silu") -> Optional[torch.Tensor]:
    """The fused kernel's result when it applies (no gradient wanted, SiLU gate, enough rows, supported shapes),
    else None: the caller then runs projection and activation separately."""
    if act != "silu" or torch.is_grad_enabled() and (x.requires_grad or w_gate_up.requires_grad):
        return None
    x2 = x.reshape(-1, x.shape[-1])
    if x2.shape[0] < GATED_MIN_ROWS or not gated_supported(x2, w_gate_up):
        return None
    return tgemm_swiglu(x2, w_gate_up).view(*x.shape[:-1], w_gate_up.shape[0] // 2)
