"""Products of a decode batch into partial sums (`dgemm` with EPI_SLAB): ragged rows, columns and depths on every tile, and the plans."""
import pytest
import torch

from areal_vllm_amd.ops import _lib as L
from areal_vllm_amd.ops import decode_gemm as dg


def _sixteenths(*shape):
    """Sums of their products are exact in fp32, in any order."""
    return (torch.randint(-2, 3, shape, device="cuda") / 16).bfloat16()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 32, 64), (31, 96, 128), (33, 1568, 192), (65, 2048, 1536), (161, 1536, 8960), (257, 544, 448),
                                   (320, 1536, 1536), (512, 5120, 2048)])
def test_partial_sums(M, N, K):
    torch.manual_seed(M)
    x, w = _sixteenths(M, K), _sixteenths(N, K)
    ref = (x.float() @ w.float().t())
    ksplit = dg.slab_plan(M, N, K)[2]
    out = torch.full((ksplit * M + 1, N), float("nan"), device="cuda")
    slab = dg.dgemm(x, w, epilogue=dg.EPI_SLAB, out=out[:-1].view(ksplit, M, N))
    assert torch.equal(slab.sum(0), ref) and out[-1].isnan().all()
    wide = torch.full((M, K + 8), float("nan"), dtype=torch.bfloat16, device="cuda")
    wide[:, :K] = x  # rows further apart than they are long
    assert torch.equal(dg.dgemm(wide[:, :K], w, epilogue=dg.EPI_SLAB), slab)
    steps = K // 64
    for ct in range(1, 6):  # every tile of these rows, in splits of all sizes, rings of two to six stages
        for mblocks in {-(-M // 256), -(-M // 96), -(-M // 32)}:
            rt = -(-(-(-M // mblocks)) // 32)
            for ks in {1, 2, min(5, steps), steps}:
                if ks > 16 or -(-steps // ks) * (ks - 1) >= steps or (mblocks - 1) * rt * 32 >= M:
                    continue
                y = torch.full((ks, M, N), float("nan"), device="cuda")
                rc = L.lib().areal_dtile_slab(L.ptr(x), L.c_int64(K), L.ptr(w), L.ptr(y), *[L.c_int(v) for v in (
                    M, N, K, ct, mblocks, ks, 2 + ct, ct & 1)], L.stream_ptr())
                assert rc == 0 and torch.equal(y.sum(0), ref), (ct, mblocks, ks)


def test_plans_have_no_empty_part():
    for M in (1, 7, 32, 33, 93, 160, 161, 255, 257, 320, 511, 512, 700):
        for N, K in ((32, 64), (128, 2048), (896, 4864), (1536, 8960), (2048, 1536), (5120, 13824), (10240, 8192)):
            ct, mblocks, ksplit = dg.slab_plan(M, N, K)
            rt = -(-(-(-M // mblocks)) // 32)
            assert 1 <= ct <= 5 and 1 <= rt <= 8 and (mblocks - 1) * rt * 32 < M <= mblocks * rt * 32
            assert 1 <= ksplit <= 24 and -(-(K // 64) // ksplit) * (ksplit - 1) < K // 64
        for F in (4, 512, 4864, 8960, 11008, 18944):
            plan = dg.swiglu_plan(M, F)
            if plan is not None:
                w, mblocks = plan
                rt = -(-(-(-M // mblocks)) // 32)
                assert w % 4 == 0 and 4 <= w <= 80 and 1 <= rt <= 8 and (mblocks - 1) * rt * 32 < M <= mblocks * rt * 32


@pytest.mark.skipif(not L.available(), reason="the kernel library is not built")
def test_refused():
    p, i, n, none = L.c_void_p(1 << 20), L.c_int, L.c_int64, L.c_void_p(0)  # never read
    call = lambda xs=64, M=8, N=64, K=64, ct=1, mb=1, ks=1, y=p: L.lib().areal_dtile_slab(
        p, n(xs), p, y, i(M), i(N), i(K), i(ct), i(mb), i(ks), i(4), i(0), none)
    assert call(K=0) == call(K=96) == call(xs=4) == call(N=6) == call(ks=0) == call(mb=0) == -1
    assert call(y=L.c_void_p(8)) == -3
    assert call(K=128, ks=3) == -4 and call(K=64 * 5, ks=4) == -4
    assert call(ct=6) == call(ct=0) == call(M=257) == -10
