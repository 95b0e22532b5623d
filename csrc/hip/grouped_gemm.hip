// Grouped GEMM for routed experts on gfx950: tokens are sorted by expert, every expert multiplies its
// contiguous slab of rows with its own weight matrix:
//     out[t, :] = x[t, :] . W[e]^T      for offsets[e] <= t < offsets[e+1]
// x [T, K] bf16 row-major, W [E, N, K] bf16 (K contiguous, the layout of nn.Linear weights), out [T, N].
// Replaces the CUTLASS grouped_gemm the reference's MoE experts call
// (realhf/impl/model/modules/moe/experts.py:195-210).
//
// Structure: one workgroup (4 waves) per output tile of 64 or 128 rows x 64 or 128 columns; a tile never straddles
// two experts (the m-tiles of an expert cover ceil(rows/TM) * TM rows, the tail rows are masked). K is walked in 64-wide
// steps through LDS with register prefetch of the next step (loads issue before the MFMA block, the LDS
// write happens after the barrier). Both operands are K-contiguous, so MFMA fragments are plain 16-byte
// LDS reads; rows are 128 bytes with the chunk swizzle  chunk ^ ((row >> 1) & 7), which makes the 16 rows
// of a ds_read_b128 lane group hit 16 different 16-byte bank slots. The product is computed transposed
// (W rows as the A operand) so that each lane ends up with 4 consecutive output columns of one token and
// stores 8 bytes at a time.
#include <stdlib.h>

#include "flash_tiles.hpp"  // swizzled 256-byte-row LDS tiles + transposed reads (weight-gradient kernel)

// Tile `id` (tiles of TM rows, numbered expert by expert) -> its expert, the tile's number there and the expert's rows;
// false behind the last tile. A lane per expert: walking 128 experts one after the other is a chain of scalar loads ahead of
// a workgroup's first tile (7 rows on 128 experts, 1536 columns, 2048 deep: 30 us a launch, now 18).
template <int TM>
DEVINL bool gg_find_tile(const int* __restrict__ offsets, int E, int id, int& e, int& tile, int& row_lo, int& row_hi) {
  const int lane = threadIdx.x & 63;
  int before = 0;  // tiles of the experts ahead of this group of 64
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int lo = offsets[min(e0 + lane, E)], hi = offsets[min(e0 + lane + 1, E)];
    const int nt = (hi - lo + TM - 1) / TM;
    int sum = nt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(sum, o, 64);
      if (lane >= o) sum += y;
    }
    const unsigned long long found = __ballot(before + sum > id);
    if (found) {
      const int i = __ffsll(found) - 1;
      e = e0 + i;
      tile = __builtin_amdgcn_readfirstlane(id - before - __shfl(sum - nt, i, 64));
      row_lo = __builtin_amdgcn_readfirstlane(__shfl(lo, i, 64));
      row_hi = __builtin_amdgcn_readfirstlane(__shfl(hi, i, 64));
      return true;
    }
    before += __shfl(sum, 63, 64);
  }
  return false;
}

DEVINL int gg_off(int row, int ch) { return row * 128 + ((ch ^ ((row >> 1) & 7)) << 4); }

// TM x TN output tile per workgroup (64 or 128 each): the four waves form a 2 x 2 grid, a wave owns a
// (TM/2) x (TN/2) block = MI x NI MFMA tiles of 32 x 32. With 128 x 128 every 16-byte LDS fragment read feeds two
// MFMAs instead of one (64 x 64: the K loop is bound by LDS reads and barriers, not by the matrix cores).
// KH = number of 64-deep sub-tiles staged per step: with 2 a step holds twice the MFMA work between the barrier
// pairs and behind every register prefetch of the next step's global loads.
// GATED: the rows are gathered on the way in (row p of the sorted order is x[src_row[p]]) and the weights are a gate half and
// an up half: the W tile takes TN / 2 columns of each, a lane's accumulators ni = 0 | 1 are a token's gate and up values of the
// same columns, and the epilogue stores silu(gate) * up (gate and up rounded to bf16 first), [T, N / 2]. For a decode step,
// where the gather and the activation are launches of their own and little else (64 / 512 rows of 2048, 8 of 128 experts
// of 768: 166 -> 158 us / 197 -> 167, 1 row 29 -> 25).
template <int TM, int TN, int KH, bool NT, bool ROT, bool GATED>
__global__ __launch_bounds__(256) void grouped_gemm_nt_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, bf16_t* __restrict__ out, const int* __restrict__ offsets, int E,
    int N, int K, int64_t w_expert_stride, int rot, const int64_t* __restrict__ src_row) {
  static_assert(!GATED || TN == 128, "a wave's two column tiles are gate and up");
  constexpr int MI = TM / 64, NI = TN / 64;
  __shared__ __attribute__((aligned(16))) char smem[KH * (TM + TN) * 128];
  char* as = smem;                  // x tile  [KH][TM rows][64 k]
  char* bs = smem + KH * TM * 128;  // W tile  [KH][TN n][64 k]

  // ---- which expert / m-tile is this block? (tiles are numbered expert by expert)
  int tile, e, row_lo, row_hi;
  if (!gg_find_tile<TM>(offsets, E, blockIdx.y, e, tile, row_lo, row_hi)) return;  // beyond the last tile (the grid is an upper bound)
  const int m0 = row_lo + tile * TM;
  const int n0 = blockIdx.x * (GATED ? TN / 2 : TN);
  const bf16_t* we = w + (size_t)e * w_expert_stride;

  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int r = lane & 31, hf = lane >> 5;
  const int wm = wid >> 1, wn = wid & 1;  // wave -> (TM/2) x (TN/2) block (tokens (TM/2)wm.., columns (TN/2)wn..)

  // cooperative loads: thread -> (row = tid >> 3 (+32 i), chunk = tid & 7). Rows past the expert's last token are not
  // fetched (their results are not stored): a decode step's expert has a handful of rows in a 64-row tile, and what the
  // launch is bound by, a CU's load path, is then left to the weights. NT: the loads of weights pass the caches by (when: at
  // the launch below).
  const int lrow = tid >> 3, lch = tid & 7;
  bf16x8 areg[KH * TM / 32] = {}, breg[KH * TN / 32];
  int64_t arow[TM / 32];  // GATED: source row of each of this thread's tile rows
  if constexpr (GATED) {
#pragma unroll
    for (int i = 0; i < TM / 32; ++i) {
      const int m = m0 + lrow + 32 * i;
      arow[i] = m < row_hi ? src_row[m] : 0;
    }
  }
  auto load = [&](int k0) {
#pragma unroll
    for (int h = 0; h < KH; ++h) {
#pragma unroll
      for (int i = 0; i < TM / 32; ++i) {
        const int m = m0 + lrow + 32 * i;
        if (m < row_hi) areg[h * (TM / 32) + i] = ld8(x + (GATED ? (size_t)arow[i] : (size_t)m) * K + k0 + 64 * h + lch * 8);
      }
#pragma unroll
      for (int i = 0; i < TN / 32; ++i) {
        const int n = GATED ? (i & 1) * (N / 2) + n0 + 32 * (i >> 1) + lrow : n0 + lrow + 32 * i;
        const bf16x8* p = reinterpret_cast<const bf16x8*>(we + (size_t)n * K + k0 + 64 * h + lch * 8);
        breg[h * (TN / 32) + i] = NT ? __builtin_nontemporal_load(p) : *p;
      }
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int h = 0; h < KH; ++h) {
#pragma unroll
      for (int i = 0; i < TM / 32; ++i)
        *reinterpret_cast<bf16x8*>(as + h * TM * 128 + gg_off(lrow + 32 * i, lch)) = areg[h * (TM / 32) + i];
#pragma unroll
      for (int i = 0; i < TN / 32; ++i)
        *reinterpret_cast<bf16x8*>(bs + h * TN * 128 + gg_off(lrow + 32 * i, lch)) = breg[h * (TN / 32) + i];
    }
  };

  f32x16 acc[MI * NI];
#pragma unroll
  for (int t = 0; t < MI * NI; ++t)
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[t][j] = 0.f;

  const int first = ROT ? k_start(e, rot, K / (64 * KH)) * (64 * KH) : 0;  // rot: at the launch
  load(first);
  for (int k0 = 0; k0 < K; k0 += 64 * KH) {
    __syncthreads();  // previous tile fully consumed
    stage();
    if (k0 + 64 * KH < K) {
      const int next = ROT ? first + k0 + 64 * KH : k0 + 64 * KH;
      load(ROT && next >= K ? next - K : next);
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 4 * KH; ++s) {
      // A operand = W rows (output columns), B operand = token rows: acc[n][m]
      bf16x8 wf[NI], xf[MI];
      const char* bt = bs + (s >> 2) * TN * 128;
      const char* at = as + (s >> 2) * TM * 128;
#pragma unroll
      for (int ni = 0; ni < NI; ++ni)
        wf[ni] = *reinterpret_cast<const bf16x8*>(bt + gg_off((TN / 2) * wn + 32 * ni + r, 2 * (s & 3) + hf));
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
        xf[mi] = *reinterpret_cast<const bf16x8*>(at + gg_off((TM / 2) * wm + 32 * mi + r, 2 * (s & 3) + hf));
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int ni = 0; ni < NI; ++ni)
          acc[mi * NI + ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[ni], xf[mi], acc[mi * NI + ni], 0, 0, 0);
    }
  }
  // ---- epilogue: lane (token = r, hf) holds columns (reg&3) + 8(reg>>2) + 4hf of each 32 x 32 tile
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    const int m = m0 + (TM / 2) * wm + 32 * mi + r;
    if constexpr (GATED) {
      if (m < row_hi) {
        bf16_t* op = out + (size_t)m * (N / 2) + n0 + 32 * wn;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          bf16x4 v;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float a = bf2f(f2bf(acc[2 * mi][4 * g + j])), u = bf2f(f2bf(acc[2 * mi + 1][4 * g + j]));
            const float sig = 1.f / (1.f + __expf(-a));
            v[j] = f2bf(a * sig * u);
          }
          *reinterpret_cast<bf16x4*>(op + 8 * g + 4 * hf) = v;
        }
      }
    } else if (m < row_hi) {
#pragma unroll
      for (int ni = 0; ni < NI; ++ni) {
        bf16_t* op = out + (size_t)m * N + n0 + (TN / 2) * wn + 32 * ni;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          bf16x4 v;
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = f2bf(acc[mi * NI + ni][4 * g + j]);
          *reinterpret_cast<bf16x4*>(op + 8 * g + 4 * hf) = v;
        }
      }
    }
  }
}

// offsets: int32 [E+1] on the device. tile_m: rows per workgroup tile, 64 or 128 (0: 128 when the experts average
// at least 256 rows, else 64 - a tile never straddles two experts, so small experts waste less with 64).
// max_tiles: host-side upper bound of sum_e ceil(rows_e / tile_m) (T / tile_m + E is always enough).
extern "C" int areal_grouped_gemm_tile_m(int T, int E, int N, int tile_m) {
  if (tile_m == 64 || tile_m == 128) return tile_m;
  return (E > 0 && T / E >= 256) ? 128 : 64;
}

// Weights past the caches: where most experts' rows are one tile, so that a weight is read once (up to 48 rows an expert on
// average: at 64 half of them are two), and where there is more than a workgroup for each of the 256 CUs: fewer wait for
// single loads, which are then slower. us from the caches / past them, cold weights: 128 experts, 1536 columns, 2048 deep,
// 7 rows 18 / 24, 32 31 / 31, 64 59 / 52, 512 164 / 149, 48 an expert 193 / 179, 64 212 / 240, 255 465 / 642; 8 experts,
// 14336 columns, 4096 deep, 1 row 32 / 48, 2 55 / 55, 4 87 / 77, 64 184 / 167; 16 of 704 columns, 1024 deep, 16 rows 9 / 12.
// Expert e's tiles start their reduction at step 13 e (k_rotation, common.hpp) while the weights are read once: by expert, so that
// what other rows chose does not change the order of a row's sums. With more rows, whose column tiles are reread from the caches,
// the common order is level or better; below 16 rows a few experts' tiles stay apart by themselves (8 rows of 8 experts, 14336
// columns, 4096 deep 75 / 87). us without / with: 128 experts, 1536 columns, 2048 deep, 64 rows 57 / 53, 512 147 / 124,
// 1600 162 / 136, 4096 173 / 150, but 8192 207 / 213, 16000 337 / 356; 64 experts, 2816 columns, 2048 deep, 512 rows 159 / 121;
// 8 experts, 4096 columns, 14336 deep, 128 rows 191 / 186 (by row tile the same within 1 us).
static bool gg_stream(int T, int E, int col_tiles) { return T <= 48l * E && (long)(T < E ? T : E) * col_tiles > 256; }

extern "C" int areal_grouped_gemm_nt(const void* x, const void* w, void* out, const int* offsets, int T,
                                     int E, int N, int K, int64_t w_expert_stride, int max_tiles, int tile_m,
                                     hipStream_t st) {
  if (T == 0 || E == 0) return 0;
  if (N % 64 != 0 || K % 64 != 0 || K < 64) return -1;
  if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) % 16 != 0) return -2;
  if (max_tiles < 1) return -3;
  const int tm = areal_grouped_gemm_tile_m(T, E, N, tile_m);
  if (max_tiles < T / tm + E) return -4;  // the caller sized its bound for another tile height
  const int tn = (N % 128 == 0) ? 128 : 64;
  dim3 grid(N / tn, max_tiles), block(256);
  // 128-deep steps (AREAL_GROUPED_GEMM_KSTEP=128) halve the barrier pairs of the large tile but cost a wave of
  // occupancy per SIMD (3 -> 2): measured 3-15 % slower on the Qwen3-MoE expert shapes, so 64 is the default
  static const int deep = [] {
    const char* e = getenv("AREAL_GROUPED_GEMM_KSTEP");
    return e && atoi(e) == 128;
  }();
  const bool stream = gg_stream(T, E, N / tn);
  const int rot = stream && T >= 16 ? k_rotation(K) : 0;
#define AREAL_GG_LAUNCH(TM_, TN_, KH_, NT_, ROT_)                                                              \
  hipLaunchKernelGGL((grouped_gemm_nt_kernel<TM_, TN_, KH_, NT_, ROT_, false>), grid, block, 0, st, (const bf16_t*)x, \
                     (const bf16_t*)w, (bf16_t*)out, offsets, E, N, K, w_expert_stride, rot, (const int64_t*)nullptr)
  if (tm == 128 && tn == 128) {
    if (deep && K % 128 == 0) AREAL_GG_LAUNCH(128, 128, 2, false, false); else AREAL_GG_LAUNCH(128, 128, 1, false, false);
  } else if (tm == 128) AREAL_GG_LAUNCH(128, 64, 1, false, false);
  else if (tn == 128) {
    if (rot) AREAL_GG_LAUNCH(64, 128, 1, true, true);
    else if (stream) AREAL_GG_LAUNCH(64, 128, 1, true, false);
    else AREAL_GG_LAUNCH(64, 128, 1, false, false);
  } else {
    if (rot) AREAL_GG_LAUNCH(64, 64, 1, true, true);
    else if (stream) AREAL_GG_LAUNCH(64, 64, 1, true, false);
    else AREAL_GG_LAUNCH(64, 64, 1, false, false);
  }
#undef AREAL_GG_LAUNCH
  return (int)hipGetLastError();
}

// out [T, N / 2] = silu(x[src_row] . gate^T) * (x[src_row] . up^T), W [E, N, K] with the gate rows ahead of the up rows; tiles of
// 64 rows: max_tiles >= T / 64 + E
extern "C" int areal_grouped_gate_up(const void* x, const int64_t* src_row, const void* w, void* out, const int* offsets, int T,
                                     int E, int N, int K, int64_t w_expert_stride, int max_tiles, hipStream_t st) {
  if (T == 0 || E == 0) return 0;
  if (N % 128 != 0 || K % 64 != 0 || K < 64) return -1;
  if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) % 16 != 0 || w_expert_stride % 8 != 0) return -2;
  if (max_tiles < T / 64 + E || max_tiles > 65535) return -3;
  const dim3 grid(N / 128, max_tiles), block(256);
  const bool stream = gg_stream(T, E, N / 128);
  const int rot = stream && T >= 16 ? k_rotation(K) : 0;
#define AREAL_GG_LAUNCH(NT_, ROT_)                                                                                \
  hipLaunchKernelGGL((grouped_gemm_nt_kernel<64, 128, 1, NT_, ROT_, true>), grid, block, 0, st, (const bf16_t*)x,   \
                     (const bf16_t*)w, (bf16_t*)out, offsets, E, N, K, w_expert_stride, rot, src_row)
  if (rot) AREAL_GG_LAUNCH(true, true);
  else if (stream) AREAL_GG_LAUNCH(true, false);
  else AREAL_GG_LAUNCH(false, false);
#undef AREAL_GG_LAUNCH
  return (int)hipGetLastError();
}

// =====================================================================================
// Input gradient of the grouped GEMM without a transposed copy of the weights:
//     dx[t, :] = dy[t, :] . W[e]          (W[e] is [R, C]: R = rows of W = columns of dy, C = columns of dx)
// Same tiling as the forward kernel (TM tokens x 128 output columns per workgroup, reduction in 64-deep steps),
// but the reduction dimension is the SLOW dimension of W: the W tile is staged as [64 r][128 c] in the swizzled
// 256-byte-row layout of flash_tiles.hpp and becomes the A operand through transposed LDS reads of the rows
// 8hf .. 8hf+7 of a 16-deep slab - the order in which the plain 16-byte row read hands the dy fragment (B operand)
// its values.
// =====================================================================================
template <int TM>
__global__ __launch_bounds__(256) void grouped_gemm_nn_kernel(
    const bf16_t* __restrict__ dy, const bf16_t* __restrict__ w, bf16_t* __restrict__ out,
    const int* __restrict__ offsets, int E, int R, int C, int64_t w_expert_stride) {
  constexpr int MI = TM / 64;
  __shared__ __attribute__((aligned(16))) char smem[TM * 128 + 64 * 256];
  char* as = smem;             // dy tile [TM tokens][64 r], 128-byte rows (gg_off)
  char* ws = smem + TM * 128;  // W tile  [64 r][128 c], 256-byte rows (swz_off)

  int tile, e, row_lo, row_hi;
  if (!gg_find_tile<TM>(offsets, E, blockIdx.y, e, tile, row_lo, row_hi)) return;
  const int m0 = row_lo + tile * TM;
  const int c0 = blockIdx.x * 128;
  const bf16_t* we = w + (size_t)e * w_expert_stride;

  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int r = lane & 31, hf = lane >> 5, gl = lane & 15, grp = lane >> 4;
  const int wm = wid >> 1, wn = wid & 1;  // wave -> tokens (TM/2) wm .., output columns 64 wn ..

  const int arow = tid >> 3, ach = tid & 7;    // dy tile: (token arow + 32 i, 16-byte chunk ach)
  const int wrow = tid >> 4, wch = tid & 15;   // W tile: (r row wrow + 16 i, 16-byte chunk wch)
  bf16x8 areg[TM / 32], wreg[4];
  auto load = [&](int r0) {
#pragma unroll
    for (int i = 0; i < TM / 32; ++i) {
      int m = m0 + arow + 32 * i;
      m = m < row_hi ? m : row_hi - 1;
      areg[i] = ld8(dy + (size_t)m * R + r0 + ach * 8);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) wreg[i] = ld8(we + (size_t)(r0 + wrow + 16 * i) * C + c0 + wch * 8);
  };
  auto stage = [&]() {
#pragma unroll
    for (int i = 0; i < TM / 32; ++i) *reinterpret_cast<bf16x8*>(as + gg_off(arow + 32 * i, ach)) = areg[i];
#pragma unroll
    for (int i = 0; i < 4; ++i) lds_row_write(ws, wrow + 16 * i, wch, wreg[i]);
  };
  f32x16 acc[MI * 2];
#pragma unroll
  for (int t = 0; t < MI * 2; ++t)
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[t][j] = 0.f;

  // LDS addresses of the fragment reads are the same every step: computed once, outside the loop
  const char* wa[4][2][2];
  const char* xa[4][MI];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
#pragma unroll
    for (int ni = 0; ni < 2; ++ni) {
      const int col = 64 * wn + 32 * ni + 16 * (grp & 1);
      wa[s][ni][0] = tr_addr(ws, 16 * s + 8 * hf, col, gl);
      wa[s][ni][1] = tr_addr(ws, 16 * s + 8 * hf + 4, col, gl);
    }
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) xa[s][mi] = as + gg_off((TM / 2) * wm + 32 * mi + r, 2 * s + hf);
  }

  load(0);
  for (int r0 = 0; r0 < R; r0 += 64) {
    __syncthreads();
    stage();
    if (r0 + 64 < R) load(r0 + 64);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      bf16x8 wf[2], xf[MI];
#pragma unroll
      for (int ni = 0; ni < 2; ++ni) wf[ni] = cat4(tr_load(wa[s][ni][0]), tr_load(wa[s][ni][1]));
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) xf[mi] = *reinterpret_cast<const bf16x8*>(xa[s][mi]);
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int ni = 0; ni < 2; ++ni)
          acc[mi * 2 + ni] = mfma32(wf[ni], xf[mi], acc[mi * 2 + ni]);
    }
  }
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    const int m = m0 + (TM / 2) * wm + 32 * mi + r;
    if (m < row_hi) {
#pragma unroll
      for (int ni = 0; ni < 2; ++ni) {
        bf16_t* op = out + (size_t)m * C + c0 + 64 * wn + 32 * ni;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          bf16x4 v;
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = f2bf(acc[mi * 2 + ni][4 * g + j]);
          *reinterpret_cast<bf16x4*>(op + 8 * g + 4 * hf) = v;
        }
      }
    }
  }
}

// dy [T, R], w [E, R, C] (C contiguous), out [T, C]; R a multiple of 64, C a multiple of 128.
extern "C" int areal_grouped_gemm_nn(const void* dy, const void* w, void* out, const int* offsets, int T, int E,
                                     int R, int C, int64_t w_expert_stride, int max_tiles, int tile_m,
                                     hipStream_t st) {
  if (T == 0 || E == 0) return 0;
  if (R % 64 != 0 || C % 128 != 0) return -1;
  if (((uintptr_t)dy | (uintptr_t)w | (uintptr_t)out) % 16 != 0) return -2;
  const int tm = areal_grouped_gemm_tile_m(T, E, C, tile_m);
  if (max_tiles < T / tm + E) return -4;
  dim3 grid(C / 128, max_tiles), block(256);
  if (tm == 128)
    hipLaunchKernelGGL(grouped_gemm_nn_kernel<128>, grid, block, 0, st, (const bf16_t*)dy, (const bf16_t*)w,
                       (bf16_t*)out, offsets, E, R, C, w_expert_stride);
  else
    hipLaunchKernelGGL(grouped_gemm_nn_kernel<64>, grid, block, 0, st, (const bf16_t*)dy, (const bf16_t*)w,
                       (bf16_t*)out, offsets, E, R, C, w_expert_stride);
  return (int)hipGetLastError();
}

// =====================================================================================
// Weight gradient of the grouped GEMM:  dW[e][n][k] = sum over the rows t of expert e of dy[t][n] * x[t][k].
// One launch for all experts (a loop of library GEMMs is launch-bound for many small experts). Grid
// (K/128, N/128 or N/256, E); workgroup = 128 x 128 or 256 x 128 tile of dW[e], four waves 2 x 2.
// The reduction runs over TOKENS, the slow dimension of both operands, so both MFMA operands are transposed LDS
// reads (ds_read_b64_tr_b16) of token-major tiles [64 tokens][128 columns] in the swizzled layout of
// flash_tiles.hpp; rows past the expert's last token are staged as zeros. fp32 accumulation, one bf16 store.
// =====================================================================================
// (fp32 gradients that are added to: tgemm_wgrad_few_kernel of train_gemm.hip.)
template <int NS>  // the tile holds NS x 128 rows of dW (columns of dy): 128 x 128 or 256 x 128
__global__ __launch_bounds__(256) void grouped_gemm_wgrad_kernel(
    const bf16_t* __restrict__ dy, const bf16_t* __restrict__ x, bf16_t* __restrict__ dw,
    const int* __restrict__ offsets, int N, int K, int64_t dw_expert_stride) {
  constexpr int YT = 64 * 256;  // bytes of one [64 tokens][128 columns] sub-tile
  __shared__ __attribute__((aligned(16))) char smem[(NS + 1) * YT];
  char* ys = smem;            // dy tile [NS][64 tokens][128 n]
  char* xs = smem + NS * YT;  // x tile  [64 tokens][128 k]
  const int e = blockIdx.z;
  const int row_lo = offsets[e], row_hi = offsets[e + 1];
  const int k0 = blockIdx.x * 128, n0 = blockIdx.y * 128 * NS;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int r = lane & 31, hf = lane >> 5, gl = lane & 15, grp = lane >> 4;
  const int wn = wid >> 1, wk = wid & 1;  // wave -> rows 64 NS wn .. of the tile, k columns 64 wk ..

  const int lrow = tid >> 4, lch = tid & 15;  // thread -> (token row lrow + 16 i, 16-byte chunk lch)
  bf16x8 yreg[4 * NS], xreg[4];
  auto load = [&](int t0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = t0 + lrow + 16 * i;
      const bool ok = t < row_hi;
      const int tc = ok ? t : row_hi - 1;
      bf16x8 b = ld8(x + (size_t)tc * K + k0 + lch * 8);
      bf16x8 a[NS];
#pragma unroll
      for (int h = 0; h < NS; ++h) a[h] = ld8(dy + (size_t)tc * N + n0 + 128 * h + lch * 8);
      if (!ok) {  // rows past the expert's last token contribute nothing
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          b[j] = (bf16_t)0.f;
#pragma unroll
          for (int h = 0; h < NS; ++h) a[h][j] = (bf16_t)0.f;
        }
      }
      xreg[i] = b;
#pragma unroll
      for (int h = 0; h < NS; ++h) yreg[NS * i + h] = a[h];
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      lds_row_write(xs, lrow + 16 * i, lch, xreg[i]);
#pragma unroll
      for (int h = 0; h < NS; ++h) lds_row_write(ys + h * YT, lrow + 16 * i, lch, yreg[NS * i + h]);
    }
  };
  constexpr int NI = 2 * NS;  // 32-row MFMA tiles of the wave along n
  f32x16 acc[NI * 2];
#pragma unroll
  for (int t = 0; t < NI * 2; ++t)
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[t][j] = 0.f;

  // LDS addresses of the transposed fragment reads: the same every step, computed once (the swizzle costs ~10
  // vector ALU operations per address, more than the MFMAs they feed if redone inside the loop)
  const char* ya[4][NI][2];
  const char* xa[4][2][2];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int col = 64 * NS * wn + 32 * i;  // row of the tile = column of dy, 0 .. 128 NS
      const int c0 = (col & 127) + 16 * (grp & 1);
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2) ya[s][i][h2] = tr_addr(ys + (col >> 7) * YT, 16 * s + 8 * h2 + 4 * hf, c0, gl);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int c0 = 64 * wk + 32 * i + 16 * (grp & 1);
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2) xa[s][i][h2] = tr_addr(xs, 16 * s + 8 * h2 + 4 * hf, c0, gl);
    }
  }

  if (row_lo < row_hi) load(row_lo);
  for (int t0 = row_lo; t0 < row_hi; t0 += 64) {
    __syncthreads();  // previous tile fully consumed
    stage();
    if (t0 + 64 < row_hi) load(t0 + 64);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 4; ++s) {  // 16-token slabs
      bf16x8 af[NI], bf[2];
#pragma unroll
      for (int i = 0; i < NI; ++i) af[i] = cat4(tr_load(ya[s][i][0]), tr_load(ya[s][i][1]));
#pragma unroll
      for (int i = 0; i < 2; ++i) bf[i] = cat4(tr_load(xa[s][i][0]), tr_load(xa[s][i][1]));
#pragma unroll
      for (int ni = 0; ni < NI; ++ni)
#pragma unroll
        for (int ki = 0; ki < 2; ++ki) acc[2 * ni + ki] = mfma32(af[ni], bf[ki], acc[2 * ni + ki]);
    }
  }
  // ---- epilogue: lane (k column = r, hf), reg -> n row (reg&3) + 8(reg>>2) + 4hf of each 32 x 32 tile
  bf16_t* de = dw + (size_t)e * dw_expert_stride;
#pragma unroll
  for (int ni = 0; ni < NI; ++ni)
#pragma unroll
    for (int ki = 0; ki < 2; ++ki) {
      bf16_t* op = de + (size_t)(n0 + 64 * NS * wn + 32 * ni + 4 * hf) * K + k0 + 64 * wk + 32 * ki + r;
#pragma unroll
      for (int reg = 0; reg < 16; ++reg) op[(size_t)((reg & 3) + 8 * (reg >> 2)) * K] = f2bf(acc[2 * ni + ki][reg]);
    }
}

// dy [T, N], x [T, K] bf16 row-major (rows sorted by expert); N and K multiples of 128; dw [E, N, K]
// bf16, every element is written (experts without rows get zeros).
extern "C" int areal_grouped_gemm_wgrad(const void* dy, const void* x, void* dw, const int* offsets, int T, int E,
                                        int N, int K, int64_t dw_expert_stride, hipStream_t st) {
  if (E == 0) return 0;
  if (N % 128 != 0 || K % 128 != 0) return -1;
  if (((uintptr_t)dy | (uintptr_t)x | (uintptr_t)dw) % 16 != 0) return -2;
  if (E > 65535 || N / 128 > 65535) return -3;
  dim3 block(256);
  // 256 x 128 tiles feed four MFMAs per transposed x fragment but hold one wave per SIMD (282 registers); the
  // 128 x 128 tile runs two and measured 3 % faster on the Qwen3-MoE shapes. AREAL_GROUPED_WGRAD_TALL=1 selects it.
  static const bool want_tall = [] { const char* e = getenv("AREAL_GROUPED_WGRAD_TALL"); return e && e[0] == '1'; }();
  const bool tall = want_tall && N % 256 == 0;
  dim3 grid(K / 128, tall ? N / 256 : N / 128, E);
  const auto kernel = tall ? grouped_gemm_wgrad_kernel<2> : grouped_gemm_wgrad_kernel<1>;
  hipLaunchKernelGGL(kernel, grid, block, 0, st, (const bf16_t*)dy, (const bf16_t*)x, (bf16_t*)dw, offsets, N, K, dw_expert_stride);
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------------------
// Grouped product for ANY operand shape and for bf16 or fp32 storage (fp32: true fp32 multiply-adds): what the
// matrix-core kernel above does not take (sizes that are no multiples of 64, fp32 serving). Workgroup (e, c) owns
// expert e and 64 output columns and walks the expert's rows in tiles of 32; operands pass through LDS in k-chunks of
// 32, every thread keeps 8 rows of one column. Row ranges come from the device, so the launch depends on shapes only.
namespace {
template <typename T> DEVINL float gg_ld(const T* p, size_t i);
template <> DEVINL float gg_ld<bf16_t>(const bf16_t* p, size_t i) { return bf2f(p[i]); }
template <> DEVINL float gg_ld<float>(const float* p, size_t i) { return p[i]; }
template <typename T> DEVINL void gg_st(T* p, size_t i, float v);
template <> DEVINL void gg_st<bf16_t>(bf16_t* p, size_t i, float v) { p[i] = f2bf(v); }
template <> DEVINL void gg_st<float>(float* p, size_t i, float v) { p[i] = v; }

template <typename T>
__global__ void __launch_bounds__(256) grouped_gemm_plain_kernel(const T* __restrict__ x, const T* __restrict__ w,
                                                                 T* __restrict__ out, const int* __restrict__ offsets,
                                                                 int N, int K) {
  __shared__ float xs[32][33];
  __shared__ float ws[64][33];
  const int e = blockIdx.x, n0 = blockIdx.y * 64, tid = threadIdx.x;
  const int col = tid & 63, rg = tid >> 6;
  const int r_lo = offsets[e], r_hi = offsets[e + 1];
  const T* we = w + (size_t)e * N * K;
  for (int r0 = r_lo; r0 < r_hi; r0 += 32) {
    float acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.f;
    for (int k0 = 0; k0 < K; k0 += 32) {
      __syncthreads();
      for (int i = tid; i < 32 * 32; i += 256) {
        const int r = i >> 5, kk = i & 31;
        xs[r][kk] = (r0 + r < r_hi && k0 + kk < K) ? gg_ld<T>(x, (size_t)(r0 + r) * K + k0 + kk) : 0.f;
      }
      for (int i = tid; i < 64 * 32; i += 256) {
        const int c = i >> 5, kk = i & 31;
        ws[c][kk] = (n0 + c < N && k0 + kk < K) ? gg_ld<T>(we, (size_t)(n0 + c) * K + k0 + kk) : 0.f;
      }
      __syncthreads();
#pragma unroll 8
      for (int kk = 0; kk < 32; ++kk) {
        const float wv = ws[col][kk];
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] += xs[rg * 8 + i][kk] * wv;
      }
    }
    if (n0 + col < N) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int r = r0 + rg * 8 + i;
        if (r < r_hi) gg_st<T>(out, (size_t)r * N + n0 + col, acc[i]);
      }
    }
  }
}
}  // namespace

// x [T, K] rows sorted by expert, w [E, N, K] contiguous, offsets [E + 1] on the device; dt 0: bf16, 1: fp32.
extern "C" int areal_grouped_gemm_plain(const void* x, const void* w, void* out, const int* offsets, int T, int E,
                                        int N, int K, int dt, hipStream_t st) {
  if (T == 0 || E == 0) return 0;
  if (N < 1 || K < 1 || E > 65535 * 32) return -1;
  const dim3 grid(E, (N + 63) / 64);
  if (dt == 0)
    hipLaunchKernelGGL(grouped_gemm_plain_kernel<bf16_t>, grid, dim3(256), 0, st, (const bf16_t*)x, (const bf16_t*)w,
                       (bf16_t*)out, offsets, N, K);
  else
    hipLaunchKernelGGL(grouped_gemm_plain_kernel<float>, grid, dim3(256), 0, st, (const float*)x, (const float*)w,
                       (float*)out, offsets, N, K);
  return (int)hipGetLastError();
}
