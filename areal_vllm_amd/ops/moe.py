"""Token routing glue of mixture-of-experts layers: rows into expert order and the weighted recombination of the
expert outputs, forward and backward as gathers (``csrc/hip/moe_ops.hip``; the token dispatchers of the reference:
``realhf/impl/model/modules/moe/token_dispatcher.py``).

`order` [T*k] is the expert-sorted order of the (token, choice) pairs (position p holds pair order[p] = t*k + j) and
`inv` [T*k] its inverse (pair t*k + j sits at position inv[t*k + j]). Every token occurs exactly k times, so the
scatter-adds of the textbook formulation (``index_add_`` for the combine, the indexing backward of ``x[tok]``) become
k-row gathers: each output row is written once, in a fixed order."""
import torch
import torch.nn.functional as F

from torch.autograd.function import once_differentiable

from . import _lib as L
from . import decode_gemm as dg
from . import train_gemm
from .norm_act import rmsnorm


def _hip_rows(t: torch.Tensor) -> bool:
    return L.use_hip(t) and t.dtype == torch.bfloat16 and t.shape[-1] % 8 == 0


def _gather_rows(src: torch.Tensor, idx: torch.Tensor, scale=None) -> torch.Tensor:
    """out[p] = scale[p] * src[idx[p]]"""
    if not _hip_rows(src):
        out = src[idx]
        return out if scale is None else out * scale.unsqueeze(-1).to(out.dtype)
    src = src.contiguous()
    out = torch.empty(idx.numel(), src.shape[1], dtype=src.dtype, device=src.device)
    L.check(L.lib().areal_moe_gather_rows(L.ptr(src), L.ptr(idx), L.ptr(scale) if scale is not None else None,
                                          L.ptr(out), L.c_int64(idx.numel()), L.c_int(src.shape[1]), L.stream_ptr()),
            "moe_gather_rows")
    return out


def _combine_rows(src: torch.Tensor, inv: torch.Tensor, w, T: int, k: int) -> torch.Tensor:
    """out[t] = sum_j w[t, j] * src[inv[t*k + j]]   (w None: plain sum)"""
    if not _hip_rows(src) or k > 16:
        g = src[inv].view(T, k, -1)
        if w is not None:
            g = g * w.view(T, k, 1).to(g.dtype)
        return g.sum(1, dtype=torch.float32).to(src.dtype)
    src = src.contiguous()
    out = torch.empty(T, src.shape[1], dtype=src.dtype, device=src.device)
    L.check(L.lib().areal_moe_combine_rows(L.ptr(src), L.ptr(inv), L.ptr(w) if w is not None else None, L.ptr(out),
                                           L.c_int64(T), L.c_int(k), L.c_int(src.shape[1]), L.stream_ptr()),
            "moe_combine_rows")
    return out


class _PermuteFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, order, inv, k, src_row=None):
        ctx.save_for_backward(inv)
        ctx.k = k
        return _gather_rows(x, order // k if src_row is None else src_row)

    @staticmethod
    def backward(ctx, dxs):
        (inv,) = ctx.saved_tensors
        k = ctx.k
        return _combine_rows(dxs.contiguous(), inv, None, inv.numel() // k, k), None, None, None, None


class _CombineFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, ys, w, order, inv):
        T, k = w.shape
        ctx.w_dtype = w.dtype
        w = w.to(ys.dtype).contiguous()
        ctx.save_for_backward(ys, w, order, inv)
        return _combine_rows(ys, inv, w, T, k)

    @staticmethod
    def backward(ctx, dout):
        ys, w, order, inv = ctx.saved_tensors
        T, k = w.shape
        dout = dout.contiguous()
        dys = dw = None
        if all(ctx.needs_input_grad[:2]) and k <= 16 and _hip_rows(ys) and _hip_rows(dout) and T > 0:
            ys = ys.contiguous()
            dys, dw = torch.empty_like(ys), torch.empty(T, k, dtype=ys.dtype, device=ys.device)
            L.check(L.lib().areal_moe_combine_bwd(L.ptr(dout), L.ptr(ys), L.ptr(inv), L.ptr(w), L.ptr(dys), L.ptr(dw), L.c_int64(T),
                                                  L.c_int(k), L.c_int(ys.shape[1]), L.stream_ptr()), "moe_combine_bwd")
            return dys, dw.to(ctx.w_dtype), None, None
        if ctx.needs_input_grad[0]:  # dys[p] = w[pair at p] * dout[token at p]
            dys = _gather_rows(dout, order // k, w.reshape(-1)[order].contiguous())
        if ctx.needs_input_grad[1]:  # dw[t, j] = <dout[t], ys[inv[t*k + j]]>
            if _hip_rows(ys):
                dw = torch.empty(T, k, dtype=ys.dtype, device=ys.device)
                L.check(L.lib().areal_moe_combine_dots(L.ptr(dout), L.ptr(ys), L.ptr(inv), L.ptr(dw), L.c_int64(T),
                                                       L.c_int(k), L.c_int(ys.shape[1]), L.stream_ptr()),
                        "moe_combine_dots")
            else:
                dw = (ys[inv].view(T, k, -1).float() * dout.float().unsqueeze(1)).sum(-1).to(w.dtype)
        return dys, (dw.to(ctx.w_dtype) if dw is not None else None), None, None


def moe_permute(x: torch.Tensor, order: torch.Tensor, inv: torch.Tensor, k: int, src_row=None) -> torch.Tensor:
    """x [T, H] -> rows in expert order [T*k, H] (row p = token order[p] // k = src_row[p] when the sort handed
    it out)."""
    return _PermuteFn.apply(x, order, inv, k, src_row)


def moe_topk(logits: torch.Tensor, k: int, norm: bool, out_dtype=torch.float32):
    """Softmax over the experts and its k largest entries per token, without autograd (serving, scoring passes):
    logits [T, E] fp32 or bf16 (the arithmetic is fp32 either way) -> (weights [T, k] in `out_dtype` - softmax
    probabilities, re-normalised over the k choices when `norm` -, expert ids int64 [T, k]), choices in descending
    order of probability. One launch on the GPU."""
    T, E = logits.shape
    if not (L.use_hip(logits) and logits.dtype in (torch.float32, torch.bfloat16) and E <= 512 and k <= min(64, E)
            and out_dtype in (torch.float32, torch.bfloat16)):
        topv, topi = torch.topk(torch.softmax(logits.float(), -1), k, -1)
        if norm:
            topv = topv / topv.sum(-1, keepdim=True)
        return topv.to(out_dtype), topi
    return _topk(logits.contiguous(), k, norm, out_dtype, False)


def _topk(logits: torch.Tensor, k: int, norm: bool, out_dtype, train: bool):
    T, E = logits.shape
    topi = torch.empty(T, k, dtype=torch.int64, device=logits.device)
    topv = torch.empty(T, k, dtype=out_dtype, device=logits.device)
    f32 = out_dtype == torch.float32
    L.check(L.lib().areal_moe_topk(L.ptr(logits), L.c_int(L.dtype_flag(logits)), L.c_int(0), L.c_int64(T), L.c_int(E),
                                   L.c_int(k), L.c_int(int(bool(norm))), L.c_int(int(train)), L.ptr(topi), L.ptr(topv) if f32 else None,
                                   None if f32 else L.ptr(topv), L.stream_ptr()), "moe_topk")
    return topv, topi


class _RouterFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w):
        ctx.save_for_backward(x, w)
        return F.linear(x, w)

    @staticmethod
    @once_differentiable
    def backward(ctx, dy):
        x, w = ctx.saved_tensors
        dx = train_gemm.dgrad(dy, w) if ctx.needs_input_grad[0] else None
        dw = None
        if ctx.needs_input_grad[1]:
            acc = torch.zeros(w.shape, dtype=torch.float32, device=w.device)
            dw = (train_gemm.tgemm_wgrad_(acc, dy, x).to(w.dtype) if train_gemm.wgrad_supported(dy, x, acc) else torch.mm(dy.t(), x))
        return dx, dw


def router_logits(x: torch.Tensor, router: torch.Tensor) -> torch.Tensor:
    """``x [T, H] @ router[E, H].T`` with gradients. Of whole 128 x 256 tiles the router's gradient is summed by the split weight-gradient
    product (16384 tokens, 128 experts of 2048: 33 us; the library, whose tiles are not split, 135 to 171) and goes on through autograd."""
    if (router.requires_grad and torch.is_grad_enabled() and router.dim() == 2 and router.shape[0] % 128 == 0 and router.shape[1] % 256 == 0
            and x.dim() == 2 and L.use_hip(x) and x.dtype == router.dtype == torch.bfloat16 and train_gemm.plain(x, router)):
        return _RouterFn.apply(x, router)
    return F.linear(x, router)


class _TopkFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, logits, k, norm):
        logits = logits.contiguous()
        topv, topi = _topk(logits, k, norm, torch.float32, True)
        ctx.save_for_backward(logits, topi)
        ctx.norm = norm
        ctx.mark_non_differentiable(topi)
        return topv, topi

    @staticmethod
    @once_differentiable
    def backward(ctx, dv, _):
        logits, topi = ctx.saved_tensors
        (T, E), k = logits.shape, topi.shape[1]
        out = torch.empty_like(logits)
        dv = dv.float().contiguous()
        L.check(L.lib().areal_moe_topk_bwd(L.ptr(logits), L.c_int(L.dtype_flag(logits)), L.c_int64(T), L.c_int(E), L.c_int(k),
                                           L.c_int(int(bool(ctx.norm))), L.ptr(topi), L.ptr(dv), L.ptr(out), L.stream_ptr()),
                "moe_topk_bwd")
        return out, None, None


def moe_topk_grad(logits: torch.Tensor, k: int, norm: bool):
    """`moe_topk` with fp32 weights that a gradient flows through: one launch each way on the GPU (its kernels serve up to 512
    experts and 64 choices of plain tensors), library operations elsewhere."""
    if (L.use_hip(logits) and logits.dtype in (torch.float32, torch.bfloat16) and logits.shape[1] <= 512 and k <= min(64, logits.shape[1])
            and logits.shape[0] > 0 and train_gemm.plain(logits)):
        return _TopkFn.apply(logits, k, norm)
    topv, topi = torch.topk(torch.softmax(logits.float(), -1), k, -1)
    return (topv / topv.sum(-1, keepdim=True) if norm else topv), topi


# Where a router's product in partial sums pays: few experts of few columns, whose tiles are few. us of the library's product / of
# partial sums, each with the top-k, cold weights, 16 / 128 / 512 rows: 32 experts, 2048 deep 11.9 / 9.0, 12.4 / 9.4, 12.7 / 10.4; 128,
# 2048 deep 12.6 / 10.7, 12.8 / 11.5, 13.3 / 12.8; 128, 4096 deep 15.6 / 12.1, 16.2 / 13.8, 16.5 / 17.1; 64, 7168 deep 12.2 / 10.9, 12.6 /
# 12.4, 13.0 / 14.4; but 128, 7168 deep 12.9 / 14.0, 14.0 / 15.3, 14.6 / 20.2; 256, 2048 deep 13.8 / 14.1, 13.9 / 14.9, 14.6 / 16.9; 512,
# 4096 deep 21.7 / 26.0, 22.0 / 27.3, 20.3 / 34.6.
ROUTE_MAX_EXPERTS, ROUTE_MAX_SIZE, ROUTE_MAX_SIZE_MANY_ROWS = 160, 1 << 19, 9 << 15


def _route_in_parts(T: int, E: int, H: int) -> bool:
    return 0 < T <= dg.MAX_ROWS and E <= ROUTE_MAX_EXPERTS and E * H <= (ROUTE_MAX_SIZE if T <= 128 else ROUTE_MAX_SIZE_MANY_ROWS)


def moe_route(x: torch.Tensor, router: torch.Tensor, k: int, norm: bool, out_dtype=torch.float32):
    """`moe_topk` of the router's projection x [T, H] @ router [E, H]^T (rounded to x's dtype). A decode batch's projection is a
    few tiles: split over the depth to fill the chip, its fp32 partial products are summed by the top-k kernel itself."""
    T, E = x.shape[0], router.shape[0]
    if not (x.is_cuda and _route_in_parts(T, E, x.shape[1]) and dg.serves(x, router) and k <= min(64, E)
            and out_dtype in (torch.float32, torch.bfloat16)):
        return moe_topk(F.linear(x, router), k, norm, out_dtype)
    slab = dg.dgemm(x, router, epilogue=dg.EPI_SLAB)
    topi = torch.empty(T, k, dtype=torch.int64, device=x.device)
    topv = torch.empty(T, k, dtype=out_dtype, device=x.device)
    f32 = out_dtype == torch.float32
    L.check(L.lib().areal_moe_topk(L.ptr(slab), L.c_int(L.dtype_flag(slab)), L.c_int(slab.shape[0]), L.c_int64(T), L.c_int(E),
                                   L.c_int(k), L.c_int(int(bool(norm))), L.c_int(0), L.ptr(topi), L.ptr(topv) if f32 else None,
                                   None if f32 else L.ptr(topv), L.stream_ptr()), "moe_topk")
    return topv, topi


def moe_group_topk(logits: torch.Tensor, k: int, n_groups: int, keep: int):
    """Sigmoid scores with group-limited choice, without autograd: logits fp32 [T, E]; the experts form `n_groups` equal
    groups of neighbours, a group's score is the sum of its two largest sigmoid scores (of its only one for groups of
    one), and the k largest scores among the members of the `keep` best groups are chosen. Returns (weights fp32 [T, k] =
    the chosen scores as they are, expert ids int64 [T, k]), choices in descending order of score. One launch on the
    GPU."""
    T, E = logits.shape
    assert logits.dtype == torch.float32 and E % n_groups == 0 and 1 <= keep <= n_groups and 1 <= k <= E
    if L.use_hip(logits) and E <= 512 and k <= 64:
        logits = logits.contiguous()
        topi = torch.empty(T, k, dtype=torch.int64, device=logits.device)
        topv = torch.empty(T, k, dtype=torch.float32, device=logits.device)
        L.check(L.lib().areal_moe_group_topk(L.ptr(logits), L.c_int64(T), L.c_int(E), L.c_int(k), L.c_int(n_groups),
                                             L.c_int(keep), L.ptr(topi), L.ptr(topv), L.stream_ptr()), "moe_group_topk")
        return topv, topi
    s = torch.sigmoid(logits)
    masked = s
    if n_groups > 1 and keep < n_groups:
        gs = E // n_groups
        grouped = s.view(T, n_groups, gs)
        gscore = grouped.topk(min(2, gs), -1).values.sum(-1)
        best = gscore.topk(keep, -1).indices
        ok = torch.zeros(T, n_groups, dtype=torch.bool, device=s.device).scatter_(1, best, True)
        masked = grouped.masked_fill(~ok.unsqueeze(-1), float("-inf")).view(T, E)
    topv, topi = masked.topk(k, -1)
    return torch.where(torch.isinf(topv), torch.zeros_like(topv), topv), topi


def moe_corrected_topk(logits: torch.Tensor, k: int, n_groups: int, keep: int, correction: torch.Tensor, scale: float):
    """Softmax scores s over all experts with a learned correction of the choice, without autograd: logits fp32 [T, E] (a
    view with unit column stride); experts are chosen by s + correction, among the members of the `keep` groups whose
    largest s + correction is largest (others count as minus infinity: the sums may be negative). Returns (weights fp32
    [T, k]: the chosen s, without the correction, divided by their sum (+ 1e-20), times `scale`; expert ids int64 [T, k]).
    One launch on the GPU."""
    T, E = logits.shape
    assert logits.dtype == torch.float32 and E % n_groups == 0 and 1 <= keep <= n_groups and 1 <= k <= E
    assert correction.numel() == E
    if L.use_hip(logits) and E <= 512 and k <= 64:
        assert logits.stride(1) == 1 and correction.is_contiguous()
        topi = torch.empty(T, k, dtype=torch.int64, device=logits.device)
        topv = torch.empty(T, k, dtype=torch.float32, device=logits.device)
        L.check(L.lib().areal_moe_corrected_topk(
            L.ptr(logits), L.c_int64(logits.stride(0)), L.c_int64(T), L.c_int(E), L.c_int(k), L.c_int(n_groups),
            L.c_int(keep), L.ptr(correction), L.c_float(scale), L.c_int(L.dtype_flag(correction)), L.ptr(topi), L.ptr(topv),
            L.stream_ptr()), "moe_corrected_topk")
        return topv, topi
    s = torch.softmax(logits, -1)
    c = s + correction.float()
    if n_groups > 1 and keep < n_groups:
        grouped = c.view(T, n_groups, E // n_groups)
        best = grouped.amax(-1).topk(keep, -1).indices
        ok = torch.zeros(T, n_groups, dtype=torch.bool, device=s.device).scatter_(1, best, True)
        c = grouped.masked_fill(~ok.unsqueeze(-1), float("-inf")).view(T, E)
    topc, topi = c.topk(k, -1)
    w = torch.where(torch.isinf(topc), torch.zeros_like(topc), s.gather(1, topi))
    return w / (w.sum(-1, keepdim=True) + 1e-20) * float(scale), topi


def moe_sort(flat_e: torch.Tensor, n_experts: int, k: int):
    """Expert-sorted order of the (token, choice) pairs: flat_e int64 [T*k] with ids 0 .. n_experts (id n_experts =
    dropped pair, sorted last) -> (order [T*k], inv [T*k], src_row [T*k] = order // k, all int64; offsets int32
    [n_experts + 2]: expert e owns positions offsets[e] .. offsets[e + 1], the dropped pairs sit from
    offsets[n_experts] on). The order is the stable one (ties in pair order), what ``torch.argsort(stable=True)``
    gives; on the GPU a counting sort in one launch (lists of a few thousand pairs: a decode batch) or three."""
    n = flat_e.numel()
    bins = n_experts + 1
    if not (L.use_hip(flat_e) and flat_e.dtype == torch.int64 and bins <= 513):
        order = torch.argsort(flat_e, stable=True)
        inv = torch.empty_like(order)
        inv[order] = torch.arange(n, device=flat_e.device)
        counts = torch.bincount(flat_e, minlength=bins)[:bins]
        offsets = torch.zeros(bins + 1, dtype=torch.int32, device=flat_e.device)
        offsets[1:] = torch.cumsum(counts, 0)
        return order, inv, order // k, offsets
    flat_e = flat_e.contiguous()
    lib = L.lib()
    order = torch.empty(n, dtype=torch.int64, device=flat_e.device)
    inv = torch.empty_like(order)
    src_row = torch.empty_like(order)
    offsets = torch.empty(bins + 1, dtype=torch.int32, device=flat_e.device)
    items, ws = 1, None
    if not int(lib.areal_moe_sort_single(L.c_int64(n), L.c_int(bins))):
        items = max(1, -(-n // (256 * 128)))  # at most 128 chunks
        chunks = -(-n // (256 * items))
        ws = torch.empty(chunks * bins, dtype=torch.int32, device=flat_e.device)
    L.check(lib.areal_moe_sort(L.ptr(flat_e), L.c_int64(n), L.c_int(bins), L.c_int(k), L.ptr(order), L.ptr(inv),
                               L.ptr(src_row), L.ptr(offsets), L.ptr(ws), L.c_int(items), L.stream_ptr()),
            "moe_sort")
    return order, inv, src_row, offsets


def host_list(t: torch.Tensor):
    """``t.tolist()`` in two halves: starts the copy and returns a function that waits for it (not for what the caller has
    launched in between)."""
    if not t.is_cuda:
        return t.tolist
    host = torch.empty(t.shape, dtype=t.dtype, pin_memory=True)
    host.copy_(t, non_blocking=True)
    done = torch.cuda.Event()
    done.record(torch.cuda.current_stream(t.device))

    def wait():
        done.synchronize()
        return host.tolist()

    return wait


def moe_combine(ys: torch.Tensor, w: torch.Tensor, order: torch.Tensor, inv: torch.Tensor) -> torch.Tensor:
    """Expert outputs in expert order ys [T*k, H], routing weights w [T, k] -> [T, H]."""
    return _CombineFn.apply(ys, w, order, inv)


def moe_combine_rmsnorm(ys: torch.Tensor, w: torch.Tensor, inv: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor,
                        eps: float, gemma: bool = False):
    """(rmsnorm(c + residual), c + residual) with c = `moe_combine` of the expert outputs, without autograd: one launch on the
    GPU."""
    T, k = w.shape
    H = ys.shape[1]
    w = w.to(ys.dtype).contiguous()
    if not (_hip_rows(ys) and 1 <= k <= 16 and H <= 8192 and ys.dtype == residual.dtype == weight.dtype
            and all(t.data_ptr() % 16 == 0 for t in (ys, residual, weight))):
        return rmsnorm(_combine_rows(ys, inv, w, T, k), weight, eps, residual, gemma)
    ys, residual, weight = ys.contiguous(), residual.contiguous(), weight.contiguous()
    y, out = torch.empty_like(residual), torch.empty_like(residual)
    L.check(L.lib().areal_moe_combine_rmsnorm(L.ptr(ys), L.ptr(inv), L.ptr(w), L.ptr(residual), L.ptr(weight), L.ptr(out),
                                              L.ptr(y), L.c_int64(T), L.c_int(k), L.c_int(H), L.c_float(eps),
                                              L.c_int(int(gemma)), L.stream_ptr()), "moe_combine_rmsnorm")
    return y, out


def clamped_glu(gu: torch.Tensor, limit: float, alpha: float = 1.702) -> torch.Tensor:
    """Gated unit with clamped pre-activations: gu [n, 2F] = gate | up ->  g sigmoid(alpha g) (u + 1)  with
    g = min(gate, limit), u = clamp(up, -limit, limit); [n, F] in gu's dtype (fp32 arithmetic)."""
    n, F2 = gu.shape
    F = F2 // 2
    if L.use_hip(gu):
        assert gu.is_contiguous()
        out = torch.empty(n, F, dtype=gu.dtype, device=gu.device)
        if n:
            L.check(L.lib().areal_clamped_glu(L.ptr(gu), L.ptr(out), L.c_int64(n), L.c_int(F), L.c_float(limit),
                                              L.c_float(alpha), L.c_int(L.dtype_flag(gu)), L.stream_ptr()),
                    "clamped_glu")
        return out
    g = gu[:, :F].float().clamp(max=limit)
    u = gu[:, F:].float().clamp(-limit, limit)
    return (g * torch.sigmoid(alpha * g) * (u + 1.0)).to(gu.dtype)


def combine_rows_w32(ys: torch.Tensor, inv: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """out[t] = sum_j w[t, j] * ys[inv[t*k + j]] with fp32 weights w [T, k] and an fp32 sum; ys [T*k, H] in expert
    order, result in ys's dtype."""
    T, k = w.shape
    assert w.dtype == torch.float32
    if L.use_hip(ys):
        ys = ys.contiguous()
        out = torch.empty(T, ys.shape[1], dtype=ys.dtype, device=ys.device)
        if T:
            L.check(L.lib().areal_moe_combine_w32(L.ptr(ys), L.ptr(inv), L.ptr(w.contiguous()), L.ptr(out),
                                                  L.c_int64(T), L.c_int(k), L.c_int(ys.shape[1]),
                                                  L.c_int(L.dtype_flag(ys)), L.stream_ptr()), "moe_combine_w32")
        return out
    return (ys[inv].view(T, k, -1).float() * w.view(T, k, 1)).sum(1).to(ys.dtype)
