// Decode-batch GEMMs for gfx950 on 16-wide tiles, with the fragments of the next half step requested while the present one is
// multiplied: Y = X W^T for M = 1 ... 512 rows, either the gated-MLP projection with its activation in the epilogue
//     Y[M, F] = act(X W_gate^T) * (X W_up^T),  W = [gate; up] [2F, K]
// or fp32 partial sums of a reduction split over workgroups, Y [ksplit, M, N], summed in split order by the row kernel that follows
// (decode_gemm.hip).
//
// What bounds these products is, in this order:
//   * the CU's load path. Loads return in order through a buffer of 32 to 64 KB: 23 GB/s a CU for bytes that come from HBM (all CUs
//     together 6 TB/s), 100 to 110 for bytes that are in the XCD's L2, 42 where the two alternate one to one and 57 one to three. A
//     workgroup stages (rows + weight rows) x K, so its rows are padded to 32 only (320 rows are two blocks of 160, not of 192) and
//     its column range has ANY width (a multiple of 4; F = 8960: 72 of 125 ranges), which gives every CU one workgroup;
//   * the matrix pipe, and LDS reads that block their wave's issue until the LDS has taken them. 2 x 2 waves, each on 16 RT rows
//     and 16 CT weight rows, read RT + CT fragments for RT x CT products (a quarter of the rows and all columns, as before: 13 reads
//     for 30 products at 192 x 72, now 10 for 25), and the reads of the next 32 deep are dealt out between the products of the
//     present ones. 64 deep at 160 x (72 + 72): 2500 cycles before; now 1125 from LDS alone, 1590 with weights from HBM.
// Captured, cold weights, us before / now: gate|up of 8960 columns, 1536 deep, 24 / 93 / 320 / 512 rows 12.8 / 12.0, 17.5 / 16.3, 29.1 /
// 24.6, 35.3 / 31.2; 14336, 4096 deep, 200 rows 71.7 / 57.3; partial sums (on decode_gemm.hip's tiles before) of 1536 columns, 8960 deep,
// 24 / 93 / 320 rows 8.2 / 7.3, 10.7 / 9.7, 21.3 / 17.4; 2048, 1536 deep 4.5 / 4.0, 5.7 / 5.2, 9.7 / 7.4; 5120, 13824 deep 29.9 / 24.9, 41.7 /
// 30.3, 76.4 / 50.6; 6144, 4096 deep 16.0 / 10.7, 19.8 / 13.7, 44.3 / 25.1. Faster at all of 156 and 97 sizes measured.
//
//   * waves 4..7 do nothing but issue the LDS-DMA pieces (global_load_lds_dwordx4, 8 rows x 128 B each) of a ring of stages, one raw
//     s_barrier per 64-deep step, counted vmcnt so that the later stages stay in flight across it; the XOR swizzle that makes the
//     ds_read_b128 fragment reads conflict-free sits on the per-lane SOURCE address;
//   * a workgroup's place by reciprocals of the host and 32-bit row products, ahead of the first load: launches of one kernel behind another
//     0.1 us each (24 rows, 1536 deep to 1536 columns 3.81 -> 3.68, 8960 deep 7.30 -> 7.19; gate|up of 320 rows 26.1 -> 25.7). Between the
//     other kernels of a step 0.2 to 0.6 at 320 rows (down 17.7 -> 17.4, gate|up 25.2 -> 24.6) and nothing at 24 (4.71 / 4.73, 7.34 / 7.60).
//   * product transposed (A = weight rows, B = activation rows). A gated block's weight tiles hold two gate rows and the two matching
//     up rows of every four, so that a lane has both factors of an output, and a pair of tiles gives it four columns in a row: an
//     8-byte store. A wave's last tile of an odd number gives two columns.
//
// Role in the reference: the MLP GEMM + activation kernels of its serving engine (areal/api/cli_args.py:398-454).
#include "common.hpp"

namespace {

typedef const __attribute__((address_space(1))) void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;

enum { DT_GATED = 0, DT_SLAB = 1 };

struct DTArgs {
  const bf16_t* X;
  long xs;
  const bf16_t* W;
  void* Y;
  long ys;
  int M, N, K;   // N: output columns (gated: F)
  int w;         // columns per range (multiple of 4)
  int ntiles;    // ceil(N / w)
  int mblocks;   // row blocks of 32 RT rows
  int ksplit, steps;  // workgroups a reduction, 64-deep steps of each (the last one's may be fewer, not 0)
  int stages;    // LDS ring
  int nt;        // non-temporal weight loads
  int act;       // gate activation: 0 SiLU (SwiGLU), 1 tanh-approximated GELU (GeGLU)
  unsigned inv_m, inv_t;  // reciprocals of mblocks and ntiles (quotient)
  int rot;       // range t starts its reduction at step t * rot and wraps round: k_rotation (common.hpp)
};

template <int N>
DEVINL void dt_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Wait until at most `keep` stages (IPW pieces of this wave each) that were issued after the one needed now are in flight.
template <int IPW>
DEVINL void dt_wait(int keep) {
  constexpr int C = 63;  // largest count the instruction encodes; a smaller count only waits for more
  switch (keep) {
    case 0: dt_vmcnt<0>(); break;
    case 1: dt_vmcnt<(IPW < C ? IPW : C)>(); break;
    case 2: dt_vmcnt<(2 * IPW < C ? 2 * IPW : C)>(); break;
    case 3: dt_vmcnt<(3 * IPW < C ? 3 * IPW : C)>(); break;
    default: dt_vmcnt<(4 * IPW < C ? 4 * IPW : C)>(); break;
  }
}

// x / (1 + exp(-x)), correctly rounded quotient (train_gemm.hip's tg_silu: a Newton step on the quotient behind v_rcp_f32).
DEVINL float dt_silu(float g) {
  const float a = 0.25f * g, d = fmaf(0.25f, __expf(-g), 0.25f);
  const float y = __builtin_amdgcn_rcpf(d), q = a * y;
  return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, a), y, q), d, a);
}
template <bool GELU>
DEVINL float dt_gate(float x) {
  if (!GELU) return dt_silu(x);
  const float inner = 0.7978845608028654f * (x + 0.044715f * x * x * x);
  const float e = __expf(-2.f * fabsf(inner));
  return 0.5f * x * (1.f + copysignf((1.f - e) / (1.f + e), inner));
}

// LDS reads may not cross this barrier; the builtin's wait tells the compiler that nothing is outstanding behind it (its own count
// would merge the loop's two read groups and wait for both before the first product).
DEVINL void dt_lds_done() { __builtin_amdgcn_s_waitcnt(0xC07F); }  // lgkmcnt(0)
DEVINL void dt_barrier() {
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int RT, int CT>
struct DTFrag {
  bf16x8 x[RT], w[CT];
  DEVINL void read(const char* xp, const char* wp) {
#pragma unroll
    for (int r = 0; r < RT; ++r) x[r] = *reinterpret_cast<const bf16x8*>(xp + r * 2048);
#pragma unroll
    for (int c = 0; c < CT; ++c) w[c] = *reinterpret_cast<const bf16x8*>(wp + c * 2048);
  }
  DEVINL void multiply(f32x4 (&acc)[CT][RT]) const {
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int r = 0; r < RT; ++r) acc[c][r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[c], x[r], acc[c][r], 0, 0, 0);
  }
};

// The reads since the last sched_barrier, dealt out between the products since then.
template <int RT, int CT, int ID>
DEVINL void dt_deal() {
  constexpr int PER = (CT * RT) / (CT + RT) > 0 ? (CT * RT) / (CT + RT) : 1;
#pragma unroll
  for (int i = 0; i < CT + RT; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x100, 1, ID);
    __builtin_amdgcn_sched_group_barrier(0x8, PER, ID);
  }
  __builtin_amdgcn_sched_group_barrier(0x8, CT * RT, ID);
  __builtin_amdgcn_sched_barrier(0);
}

// A wave's gated outputs: rows m + 16 r, columns from nb on, below c1. All of a row's values are computed before the first store: in
// the branches of the stores, four at a time and with the compiler's division, 50 outputs a lane took 8500 cycles; now 5060.
template <int RT, int CT, bool GELU>
DEVINL void dt_store_gated(const DTArgs& a, const f32x4 (&acc)[CT][RT], int m, int nb, int c1, int q) {
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    bf16x2 o[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int j = 0; j < 2; ++j)  // gate / up rounded to bf16 first: the values an unfused bf16 GEMM output would carry
        o[c][j] = f2bf(dt_gate<GELU>(bf2f(f2bf(acc[c][r][j]))) * bf2f(f2bf(acc[c][r][2 + j])));
    if (m + 16 * r >= a.M) continue;
    bf16_t* y = (bf16_t*)a.Y + (size_t)(m + 16 * r) * a.ys;
#pragma unroll
    for (int p = 0; p < CT / 2; ++p) {
      const int n = nb + 16 * p + 4 * q;  // ranges and this wave's part start at multiples of 4: the four columns are inside together
      if (n < c1) *reinterpret_cast<bf16x4*>(y + n) = bf16x4{o[2 * p][0], o[2 * p][1], o[2 * p + 1][0], o[2 * p + 1][1]};
    }
    if constexpr (CT & 1) {
      const int n = nb + 8 * (CT - 1) + 2 * q;
      if (n < c1) *reinterpret_cast<bf16x2*>(y + n) = o[CT - 1];
    }
  }
}

template <int RT, int CT, int EPI, bool ROT>
__global__ __launch_bounds__(512) void dtile_kernel(const DTArgs a) {
  constexpr int BM = 32 * RT, WR = 32 * CT;  // activation rows and weight rows of a stage
  constexpr int IPW = RT + CT;               // 1-KiB pieces per stage and loader wave
  constexpr int STAGE_BYTES = (BM + WR) * 128;
  // both halves' fragments beside the accumulators of large tiles exceed the 256 registers of a wave
  constexpr bool AHEAD = 4 * RT * CT + 8 * (RT + CT) <= 224;
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Ids are dealt round-robin to the 8 XCDs: each XCD takes a contiguous range, row blocks first, then column ranges, then splits, so
  // that a weight range's row blocks meet in one L2 and a slice of X is fetched by one or two of them.
  int tile, mb, sp;
  {
    const int nb = gridDim.x, q = nb >> 3, r = nb & 7, x = blockIdx.x & 7;
    const int pos = (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + (blockIdx.x >> 3);
    const int rest = quotient(pos, a.mblocks, a.inv_m);
    mb = pos - rest * a.mblocks;
    sp = quotient(rest, a.ntiles, a.inv_t);
    tile = rest - sp * a.ntiles;
  }
  const int c0 = tile * a.w;
  const int c1 = min(a.N, c0 + a.w);
  const int m0 = mb * BM;
  const int k0 = sp * a.steps * 64;
  const int nsteps = min(a.steps, (a.K >> 6) - sp * a.steps);
  const int stages = a.stages;

  if (wave >= 4) {
    // ---- staging: piece i of a stage = LDS rows 8i .. 8i+7 (weight rows, then activation rows); this wave has every fourth
    const int lw = wave - 4;
    const bf16_t* src[IPW];
#pragma unroll
    for (int j = 0; j < IPW; ++j) {
      const int row = 8 * (lw + 4 * j) + (lane >> 3);
      const int c = (lane & 7) ^ ((row >> 1) & 7);  // logical 16-byte chunk stored at physical chunk lane&7
      if (j < CT) {
        size_t n;  // surplus rows of the last tiles repeat the range's last column
        if (EPI == DT_GATED) {
          const int t = row >> 4, i = row & 3, q = (row & 15) >> 2, wn = t / CT, ct = t % CT;
          int col = wn * CT * 8 + 8 * (ct & ~1) + (i & 1);
          col += (CT & 1) && ct == CT - 1 ? 2 * q : 4 * q + 2 * (ct & 1);
          n = (size_t)(i >> 1) * a.N + min(c0 + col, c1 - 1);
        } else {
          n = min(c0 + row, c1 - 1);
        }
        src[j] = a.W + n * a.K + k0 + 8 * c;
      } else {
        const unsigned m = min(m0 + row - WR, a.M - 1);
        size_t at = (size_t)m * (unsigned)a.xs;  // (32 by 32 bits: a 64-bit product is four slow instructions a piece)
        if (a.xs >> 32) at += (size_t)(m * (unsigned)(a.xs >> 32)) << 32;
        src[j] = a.X + at + k0 + 8 * c;
      }
    }
    const int rot = ROT ? k_start(tile, a.rot, nsteps) : 0;
    auto issue = [&](int buf, int step) {
      if (ROT) {
        step += rot;
        step -= step >= nsteps ? nsteps : 0;
      }
      char* base = smem + buf * STAGE_BYTES + lw * 1024;
#pragma unroll
      for (int j = 0; j < IPW; ++j) {
        if (j < CT && a.nt)
          __builtin_amdgcn_global_load_lds((gptr_t)(src[j] + step * 64), (lptr_t)(base + j * 4096), 16, 0, 2);
        else
          __builtin_amdgcn_global_load_lds((gptr_t)(src[j] + step * 64), (lptr_t)(base + j * 4096), 16, 0, 0);
      }
    };
    for (int s = 0; s < stages - 1; ++s)
      if (s < nsteps) issue(s, s);
    int buf = stages - 1;
    for (int t = 0; t < nsteps; ++t) {
      dt_wait<IPW>(min(nsteps - 1 - t, stages - 2));
      __builtin_amdgcn_s_barrier();  // stage t is there, and every wave is done with stage t - 1
      if (t + stages - 1 < nsteps) {
        issue(buf, t + stages - 1);
        buf = buf + 1 == stages ? 0 : buf + 1;
      }
    }
    return;
  }

  // ---- consumers: wave (wm, wn) owns rows [16 RT wm, + 16 RT) and weight rows [16 CT wn, + 16 CT) of the stage
  const int wm = wave & 1, wn = wave >> 1;
  const int r16 = lane & 15, q = lane >> 4;
  const int key = (r16 >> 1) & 7;  // tile bases are multiples of 16 rows: the row's swizzle key is the lane's
  const int co0 = (q ^ key) << 4, co1 = ((4 + q) ^ key) << 4;
  const int wb = (wn * CT * 16 + r16) * 128, xb = (WR + wm * RT * 16 + r16) * 128;

  f32x4 acc[CT][RT];
#pragma unroll
  for (int c = 0; c < CT; ++c)
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[c][r] = f32x4{0.f, 0.f, 0.f, 0.f};

  const char* sb = smem;
  int buf = 0;
  if constexpr (AHEAD) {
    DTFrag<RT, CT> fa, fb;
    dt_barrier();
    fa.read(sb + xb + co0, sb + wb + co0);
    for (int t = 0; t + 1 < nsteps; ++t) {
      dt_lds_done();
      fb.read(sb + xb + co1, sb + wb + co1);
      fa.multiply(acc);
      dt_deal<RT, CT, 0>();
      dt_lds_done();  // every read of this stage has returned before any wave may restage it
      dt_barrier();
      buf = buf + 1 == stages ? 0 : buf + 1;
      sb = smem + buf * STAGE_BYTES;
      fa.read(sb + xb + co0, sb + wb + co0);
      fb.multiply(acc);
      dt_deal<RT, CT, 1>();
    }
    fb.read(sb + xb + co1, sb + wb + co1);
    fa.multiply(acc);
    fb.multiply(acc);
  } else {
    for (int t = 0; t < nsteps; ++t) {
      dt_barrier();
      DTFrag<RT, CT> f;
      f.read(sb + xb + co0, sb + wb + co0);
      f.multiply(acc);
      f.read(sb + xb + co1, sb + wb + co1);
      f.multiply(acc);
      dt_lds_done();
      buf = buf + 1 == stages ? 0 : buf + 1;
      sb = smem + buf * STAGE_BYTES;
    }
  }

  // ---- epilogue. acc[c][r][i]: activation row m, weight row 4 q + i of tile c
  if constexpr (EPI == DT_GATED) {
    if (a.act == 0) dt_store_gated<RT, CT, false>(a, acc, m0 + wm * RT * 16 + r16, c0 + wn * CT * 8, c1, q);
    else dt_store_gated<RT, CT, true>(a, acc, m0 + wm * RT * 16 + r16, c0 + wn * CT * 8, c1, q);
  } else {
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const int m = m0 + (wm * RT + r) * 16 + r16;
      if (m >= a.M) continue;
      float* y = (float*)a.Y + ((size_t)sp * a.M + m) * a.ys;
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        const int n = c0 + (wn * CT + c) * 16 + 4 * q;
        if (n < c1) *reinterpret_cast<f32x4*>(y + n) = acc[c][r];
      }
    }
  }
}

// Y [M, N] bf16 = X W^T for so many columns that every CU has several ranges (the LM head): as above, with a workgroup a CU that goes
// from range to range. The loader waves ask for the next range's first stages while the last ones of the present are multiplied and its
// outputs stored: with a workgroup a range the ring is empty at the start of each and drains at its end.
// us, cold weights, decode_gemm.hip's tiles / library / this: 151936 columns, 1536 deep, 96 / 128 / 160 rows 188 / 198 / -, 120 / 128 / 138, 103 /
// 111 / 119; 2048 deep 96 / 160 rows 238 / -, 161 / 181, 128 / 150; 128256, 4096 deep, 160 rows - / 249 / 229; 32000, 2048 deep, 160 rows
// - / 38 / 38. What bounds it: the X that every range stages again. All rows are one block: in two blocks (each range twice) 224 rows of the
// first took 186 where the library takes 152, 320 rows 187 / 188. Up to 64 rows a step was as long on decode_gemm.hip's tiles.
template <int RT, int CT>
__global__ __launch_bounds__(512) void dtile_walk_kernel(const DTArgs a) {
  constexpr int BM = 32 * RT, WR = 32 * CT, IPW = RT + CT;
  constexpr int STAGE_BYTES = (BM + WR) * 128;
  static_assert(4 * RT * CT + 8 * (RT + CT) <= 224, "accumulators and two sets of fragments in 256 registers");
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // in every round an XCD has neighbouring ranges
  const int nwg = gridDim.x, all = a.ntiles;
  const int first = (blockIdx.x & 7) * (nwg >> 3) + (blockIdx.x >> 3);  // (the grid is a multiple of 8)
  const int nsteps = a.K >> 6, stages = a.stages;
  const int mine = first < all ? (all - first + nwg - 1) / nwg : 0, total = mine * nsteps;

  if (wave >= 4) {
    const int lw = wave - 4;
    const bf16_t* src[IPW];
    int tile = first - nwg, step = nsteps, k = 0;
    auto issue = [&](int buf) {
      if (step == nsteps) {
        tile += nwg;
        step = 0;
        const int c0 = tile * a.w, c1 = min(a.N, c0 + a.w);
        k = k_start(tile, a.rot, nsteps);
#pragma unroll
        for (int j = 0; j < IPW; ++j) {
          const int row = 8 * (lw + 4 * j) + (lane >> 3);
          const int c = (lane & 7) ^ ((row >> 1) & 7);
          src[j] = j < CT ? a.W + (size_t)min(c0 + row, c1 - 1) * a.K + 8 * c
                          : a.X + (size_t)min(row - WR, a.M - 1) * a.xs + 8 * c;
        }
      }
      char* base = smem + buf * STAGE_BYTES + lw * 1024;
#pragma unroll
      for (int j = 0; j < IPW; ++j) {
        if (j < CT)  // weights past the caches
          __builtin_amdgcn_global_load_lds((gptr_t)(src[j] + k * 64), (lptr_t)(base + j * 4096), 16, 0, 2);
        else
          __builtin_amdgcn_global_load_lds((gptr_t)(src[j] + k * 64), (lptr_t)(base + j * 4096), 16, 0, 0);
      }
      ++step;
      k = k + 1 == nsteps ? 0 : k + 1;
    };
    for (int s = 0; s < stages - 1; ++s)
      if (s < total) issue(s);
    int buf = stages - 1;
    for (int t = 0; t < total; ++t) {
      dt_wait<IPW>(min(total - 1 - t, stages - 2));
      __builtin_amdgcn_s_barrier();  // stage t is there, and every wave is done with stage t - 1
      if (t + stages - 1 < total) {
        issue(buf);
        buf = buf + 1 == stages ? 0 : buf + 1;
      }
    }
    return;
  }

  const int wm = wave & 1, wn = wave >> 1;
  const int r16 = lane & 15, q = lane >> 4;
  const int key = (r16 >> 1) & 7;
  const int co0 = (q ^ key) << 4, co1 = ((4 + q) ^ key) << 4;
  const int wb = (wn * CT * 16 + r16) * 128, xb = (WR + wm * RT * 16 + r16) * 128;

  const char* sb = smem;
  int buf = 0;
  DTFrag<RT, CT> fa, fb;
  if (mine > 0) {
    dt_barrier();
    fa.read(sb + xb + co0, sb + wb + co0);
  }
  for (int i = 0, tile = first; i < mine; ++i, tile += nwg) {
    f32x4 acc[CT][RT];
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int r = 0; r < RT; ++r) acc[c][r] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int t = 0; t + 1 < nsteps; ++t) {
      dt_lds_done();
      fb.read(sb + xb + co1, sb + wb + co1);
      fa.multiply(acc);
      dt_deal<RT, CT, 0>();
      dt_lds_done();
      dt_barrier();
      buf = buf + 1 == stages ? 0 : buf + 1;
      sb = smem + buf * STAGE_BYTES;
      fa.read(sb + xb + co0, sb + wb + co0);
      fb.multiply(acc);
      dt_deal<RT, CT, 1>();
    }
    dt_lds_done();
    fb.read(sb + xb + co1, sb + wb + co1);
    fa.multiply(acc);
    dt_deal<RT, CT, 2>();
    dt_lds_done();
    if (i + 1 < mine) {  // on to the next range's first stage: the loaders go on while this one's outputs are stored
      dt_barrier();
      buf = buf + 1 == stages ? 0 : buf + 1;
      sb = smem + buf * STAGE_BYTES;
      fa.read(sb + xb + co0, sb + wb + co0);
    }
    fb.multiply(acc);
    const int m0 = wm * RT * 16 + r16, n0 = tile * a.w + wn * CT * 16 + 4 * q, c1 = min(a.N, tile * a.w + a.w);
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      if (m0 + 16 * r >= a.M) continue;
      bf16_t* y = (bf16_t*)a.Y + (size_t)(m0 + 16 * r) * a.ys;
#pragma unroll
      for (int c = 0; c < CT; ++c)
        if (n0 + 16 * c < c1)
          *reinterpret_cast<bf16x4*>(y + n0 + 16 * c) = bf16x4{f2bf(acc[c][r][0]), f2bf(acc[c][r][1]), f2bf(acc[c][r][2]), f2bf(acc[c][r][3])};
    }
  }
}

template <int RT, int CT>
int dt_walk(DTArgs a, int workgroups, hipStream_t st) {
  constexpr int stage_bytes = 32 * (RT + CT) * 128;
  a.stages = min(6, 160 * 1024 / stage_bytes);
  auto kern = dtile_walk_kernel<RT, CT>;
  static bool attr_set = false;  // per instantiation
  if (!attr_set) {
    HIP_RET(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 / stage_bytes * stage_bytes));
    attr_set = true;
  }
  hipLaunchKernelGGL(kern, dim3(workgroups), dim3(512), a.stages * stage_bytes, st, a);
  return (int)hipGetLastError();
}

template <int RT, int CT, int EPI, bool ROT>
int dt_launch_as(DTArgs a, hipStream_t st) {
  constexpr int stage_bytes = 32 * (RT + CT) * 128;
  a.stages = max(2, min(a.stages, min(6, 160 * 1024 / stage_bytes)));
  auto kern = dtile_kernel<RT, CT, EPI, ROT>;
  if (a.stages * stage_bytes > 64 * 1024) {
    static bool attr_set = false;  // per instantiation
    if (!attr_set) {
      HIP_RET(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 / stage_bytes * stage_bytes));
      attr_set = true;
    }
  }
  a.inv_m = reciprocal((long)a.ntiles * a.ksplit * a.mblocks, a.mblocks);
  a.inv_t = reciprocal((long)a.ntiles * a.ksplit, a.ntiles);
  hipLaunchKernelGGL(kern, dim3(a.ntiles * a.ksplit * a.mblocks), dim3(512), a.stages * stage_bytes, st, a);
  return (int)hipGetLastError();
}

template <int RT, int CT, int EPI>
int dt_launch(const DTArgs& a, hipStream_t st) {
  if constexpr (EPI == DT_GATED)
    if (a.rot) return dt_launch_as<RT, CT, EPI, true>(a, st);
  return dt_launch_as<RT, CT, EPI, false>(a, st);
}

template <int RT, int EPI>
int dt_cols(const DTArgs& a, int ct, hipStream_t st) {
  switch (ct) {
    case 1: return dt_launch<RT, 1, EPI>(a, st);
    case 2: return dt_launch<RT, 2, EPI>(a, st);
    case 3: return dt_launch<RT, 3, EPI>(a, st);
    case 4: return dt_launch<RT, 4, EPI>(a, st);
    case 5: return dt_launch<RT, 5, EPI>(a, st);
  }
  return -10;
}

template <int EPI>
int dt_rows(const DTArgs& a, int rt, int ct, hipStream_t st) {
  switch (rt) {
    case 1: return dt_cols<1, EPI>(a, ct, st);
    case 2: return dt_cols<2, EPI>(a, ct, st);
    case 3: return dt_cols<3, EPI>(a, ct, st);
    case 4: return dt_cols<4, EPI>(a, ct, st);
    case 5: return dt_cols<5, EPI>(a, ct, st);
    case 6: return dt_cols<6, EPI>(a, ct, st);
    case 7: return dt_cols<7, EPI>(a, ct, st);
    case 8: return dt_cols<8, EPI>(a, ct, st);
  }
  return -10;
}

}  // namespace

// X [M, K] bf16 (row stride xs), W = [gate; up] [2F, K] bf16 contiguous, Y [M, F] bf16 (row stride ys).
// K % 64 == 0, F % 4 == 0, w % 4 == 0, 4 <= w <= 80, M <= 256 mblocks, mblocks in {1 .. 4}. Returns -10 for a shape
// no instantiation covers (the caller then takes another kernel).
extern "C" int areal_dswiglu(const void* X, long xs, const void* W, void* Y, long ys, int M, int F, int K, int w,
                             int mblocks, int stages, int nt, int act, hipStream_t st) {
  if (M <= 0) return 0;
  if (K % 64 != 0 || K < 64 || xs % 8 != 0 || F % 4 != 0 || w % 4 != 0 || w < 4 || ys % 4 != 0) return -1;
  if (mblocks < 1 || mblocks > 4) return -2;
  if (((uintptr_t)X | (uintptr_t)W) % 16 != 0 || ((uintptr_t)Y) % 8 != 0) return -3;
  DTArgs a;
  a.X = (const bf16_t*)X; a.xs = xs; a.W = (const bf16_t*)W; a.Y = Y; a.ys = ys;
  a.M = M; a.N = F; a.K = K; a.w = w; a.ntiles = (F + w - 1) / w; a.mblocks = mblocks; a.ksplit = 1; a.steps = K / 64;
  a.stages = stages; a.nt = nt; a.act = act;
  // us without / with, 14336 columns, 4096 deep, 8 / 64 / 128 / 200 rows: 46 / 41, 47 / 41, 53 / 52, 78 / 77; 8 / 100 rows, 8192 columns
  // 34 / 25, 38 / 33, but 4096 columns 23.7 / 23.9, 30.1 / 31.0
  a.rot = mblocks == 1 && F >= 8192 ? k_rotation(K) : 0;
  const int rows = (M + mblocks - 1) / mblocks;  // rows per block
  return dt_rows<DT_GATED>(a, (rows + 31) / 32, (w + 15) / 16, st);
}

// X [M, K] bf16 (row stride xs), W [N, K] bf16 contiguous, Y fp32 [ksplit, M, N]: partial sums of 64-deep steps [s, s + 1) * steps,
// steps = ceil(K / 64 / ksplit), none of them empty. K % 64 == 0, N % 4 == 0; 32 rt rows (1 <= rt <= 8) and 32 ct columns (1 <= ct <=
// 5) a workgroup, rt >= ceil(M / 32 / mblocks).
extern "C" int areal_dtile_slab(const void* X, long xs, const void* W, void* Y, int M, int N, int K, int ct, int mblocks, int ksplit,
                                int stages, int nt, hipStream_t st) {
  if (M <= 0) return 0;
  if (K % 64 != 0 || K < 64 || xs % 8 != 0 || N % 4 != 0 || N < 4 || ksplit < 1 || mblocks < 1) return -1;
  if (((uintptr_t)X | (uintptr_t)W | (uintptr_t)Y) % 16 != 0) return -3;
  DTArgs a;
  a.X = (const bf16_t*)X; a.xs = xs; a.W = (const bf16_t*)W; a.Y = Y; a.ys = N;
  a.M = M; a.N = N; a.K = K; a.w = 32 * ct; a.mblocks = mblocks; a.ksplit = ksplit; a.steps = (K / 64 + ksplit - 1) / ksplit;
  if ((long)a.steps * (ksplit - 1) >= K / 64) return -4;  // an empty split
  if (ct < 1 || ct > 5) return -10;
  a.ntiles = (N + a.w - 1) / a.w;
  a.stages = stages; a.nt = nt; a.act = 0; a.rot = 0;
  const int rows = (M + mblocks - 1) / mblocks;
  return dt_rows<DT_SLAB>(a, (rows + 31) / 32, ct, st);
}

// X [M, K] bf16 (row stride xs), W [N, K] bf16 contiguous, Y [M, N] bf16 (row stride ys): K % 64 == 0, N % 4 == 0, 4 <= w <= 160 columns
// a range (a multiple of 4), 65 to 160 rows.
extern "C" int areal_dtile_rows(const void* X, long xs, const void* W, void* Y, long ys, int M, int N, int K, int w, int workgroups,
                                hipStream_t st) {
  if (M <= 0) return 0;
  if (K % 64 != 0 || K < 64 || xs % 8 != 0 || N % 4 != 0 || N < 4 || w % 4 != 0 || w < 4 || w > 160 || ys % 4 != 0) return -1;
  if (workgroups < 8 || workgroups % 8 != 0) return -2;
  if (((uintptr_t)X | (uintptr_t)W) % 16 != 0 || (uintptr_t)Y % 8 != 0) return -3;
  DTArgs a = {};
  a.X = (const bf16_t*)X; a.xs = xs; a.W = (const bf16_t*)W; a.Y = Y; a.ys = ys;
  a.M = M; a.N = N; a.K = K; a.w = w; a.ntiles = (N + w - 1) / w; a.rot = k_rotation(K);
  if ((long)a.ntiles * (K / 64) >= (1l << 31)) return -4;
  switch ((M + 31) / 32) {
    case 3: return dt_walk<3, 5>(a, workgroups, st);
    case 4: return dt_walk<4, 5>(a, workgroups, st);
    case 5: return dt_walk<5, 5>(a, workgroups, st);
  }
  return -10;
}
