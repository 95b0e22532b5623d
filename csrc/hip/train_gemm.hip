// Dense bf16 GEMM of the trainer and of prefill on gfx950:
//
//     C[M, N] = A[M, K] . B[N, K]^T (+ bias[N])          bf16 operands, fp32 accumulation, bf16 result
//
// Both operands are K-contiguous: A = activations, B = an nn.Linear weight; the NN form (input gradient) takes B [K, N] as the
// weight lies in memory. Role in the reference: the cuBLAS GEMMs behind torch.nn.functional.linear in
// realhf/impl/model/parallelism/tensor_parallel/modules.py:242-402 and the HF model code.
//
// Structure (one workgroup = one 256 x 256 output tile, 8 waves as 2 (M) x 4 (N), a wave owns 128 x 64):
//   * K is walked in 64-deep tiles through two LDS buffers of 64 KiB. A tile is staged as four 16-KiB PIECES
//     (128 rows x 128 B each), chosen by WHEN they are read, not by where they sit in the matrix:
//       A0 = rows 0-63 of both wave rows, A1 = rows 64-127 of both wave rows,
//       B0 = columns 0-31 of all four wave columns, B1 = columns 32-63 of all four wave columns.
//   * a K tile is four phases, each one quadrant (64 x 32) of the wave's output = 16 MFMA 16x16x32:
//       phase 1 reads B0 + A0 (12 ds_read_b128), phase 2 reads B1 (4), phase 3 reads A1 (8), phase 4 reads nothing.
//     Every phase also issues the LDS-DMA (global_load_lds_dwordx4, two per thread) of ONE piece, as soon as the piece
//     it overwrites has been read by everyone:
//       phase 1 -> A1 of tile t+1, phase 2 -> B0 of t+2, phase 3 -> A0 of t+2, phase 4 -> B1 of t+2.
//     One counted wait per tile (phase 4: vmcnt(6) = the three newest pieces may still be in flight) makes tile t+1
//     complete; it is read from the next phase on. Loads are never drained inside the loop.
//   * raw s_barrier pairs around each MFMA cluster (s_setprio keeps hipcc from moving MFMAs across them); the waves of the
//     second wave row run one barrier behind the first, so that one group's LDS reads and DMA issue overlap the other
//     group's MFMA cluster (the two groups share every SIMD).
//   * LDS rows are 128 B; the XOR swizzle chunk ^ ((row >> 1) & 7) makes every 16-lane group of a ds_read_b128 hit 16
//     different 16-byte slots. The DMA writes LDS linearly (wave base + lane x 16), so the swizzle sits on the per-lane
//     SOURCE address and on the read address.
//   * the product is computed transposed (B rows as the MFMA A operand): a lane ends up with 4 consecutive output
//     columns of one row. Results pass through the 32 KiB of LDS that the operand tiles leave free and leave as 16-byte pieces
//     of whole 128-byte lines; the gated form, whose wave has half a line, stores 16 bytes a lane from the registers.
//   * block id -> tile: contiguous id ranges per XCD (ids are dealt round-robin to the 8 XCDs), walked in bands of 4
//     tile rows so that the blocks running together on an XCD share A and B panels in its L2.
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include <hip/amd_detail/amd_hip_unsafe_atomics.h>

#include "flash_tiles.hpp"  // swizzled 256-byte-row LDS tiles + transposed reads (weight-gradient kernel)

namespace {

typedef const __attribute__((address_space(1))) void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;

struct TGArgs {
  const bf16_t* A;
  long lda;
  const bf16_t* B;
  long ldb;
  bf16_t* C;
  long ldc;
  const bf16_t* bias;
  int M, N, K;
  int tiles_m, tiles_n;
  // plain and NN: the tiles from `whole` on are reduced in `splits` parts of `chunk` 128-deep pairs each (the last one may get fewer);
  // part [splits][tile - whole][256][256] fp32
  float* part;
  int whole, splits, chunk;
  // grouped (GRP): rows sorted by expert, B [experts][..] `stride` elements apart; table[0] = row tiles of all experts, then
  // one entry {first row, end of the expert's rows, expert} a row tile, written by tgemm_table_kernel
  const int4* table;
  long stride;
  // statistics (EPI 2): log2(e) / temperature; part = [maximum | sum | weighted sum][ceil(N / 64)][M]
  float scale;
};
typedef const __attribute__((address_space(4))) int4* tg_table_t;  // scalar loads

constexpr int TG_PIECE = 128 * 128;   // bytes of one staged piece
constexpr int TG_BUF = 4 * TG_PIECE;  // A0 A1 B0 B1 of one K tile
constexpr int TG_LDS = 2 * TG_BUF;
constexpr int TG_OUT = 32 * 1024;  // the rest of the CU's 160 KiB: results on their way to whole lines
enum { PA0 = 0, PA1 = 1, PB0 = 2, PB1 = 3 };
constexpr int TG_GROUP_M = 4;

template <int N>
DEVINL void tg_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
DEVINL void tg_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Transposed LDS read, from inline assembly: behind the builtin, hipcc cannot tell it from the pending LDS-DMA writes and puts
// s_waitcnt vmcnt(0) in front of every group of reads, draining the pipeline. The results are ordered by the explicit lgkmcnt
// waits of the phase.
DEVINL bf16x4 tg_tr(uint32_t adr, int imm) {
  bf16x4 v;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(adr), "i"(imm));
  return v;
}

// gg / (1 + exp(-gg)) of a gate that was rounded to bf16, 64 of them a lane and tile. v_rcp_f32 is off by up to one step and gives 0
// where the result would be subnormal; one Newton step on the quotient (P. Markstein, IBM J. Res. Dev. 34, 1990) makes it the
// correctly rounded one: of all divisors of 24 bits, dividends of 8 and starts within a step of the reciprocal, 21 of 3.2e9 end
// a step beside it. A quarter of numerator and denominator keeps the reciprocal normal up to the largest finite exponential;
// v_div_fixup_f32 is for infinities. us at 32768 x 8960 from 1536 deep: 1321; the reciprocal alone 1292, the compiler's division 1386.
DEVINL float tg_silu(float gg) {
  const float a = 0.25f * gg, d = fmaf(0.25f, __expf(-gg), 0.25f);
  const float y = __builtin_amdgcn_rcpf(d), q = a * y;
  return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, a), y, q), d, a);
}

typedef bf16x8 tg_bfrag[2][2];  // [n tile][k step]
typedef f32x4 tg_acc[4][2];     // [m tile][n tile] of one quadrant

// EPI 0: C = A.B^T (+ bias), output tiles of 256 x 256. EPI 1 (gated MLP, no-grad forward): B = [gate rows; up rows]
// of width N each, C[M, N] = silu(A.gate^T) * (A.up^T); an output tile is 256 rows x 128 columns, its B pieces hold
// the 128 gate rows (read in the phases of the first column half) and the 128 matching up rows (second half), so a
// lane finds gate and up of the same output element in the same registers of the two accumulator quadrants.
//
// Result stores of the plain form. A lane of the MFMA result owns 4 consecutive columns of one row; stored from there, a wave
// instruction touches 16 rows and hands the memory system quarter lines: the 1.17 GB of a 32768 x 17920 result cost 320 of
// 1510 us (no stores at all: 1190). So a row half passes through the 32 KiB of LDS that the operand tiles leave free, a wave's
// own 4 KiB at a time, and leaves as whole 128-byte lines: 1510 -> 1346 us, streamed past the caches (nontemporal) 1299;
// 8192 x 151936 from 1536 deep 3287 -> 2801 us (library: 1294 and 3002). The waits of the stream do not matter: with counts
// raised by the stores in flight, so that no wait stands behind one, the times are the same.
// What is left is power: the matrix cores are busy 65 to 86 % of the time in the large products, at clocks of 1.3 to 1.8 GHz (2.4
// nominal); bare products of normal numbers reach 1.7 to 1.8 PFLOP/s on the whole chip with either instruction, of zeros 2.2 to 2.5.
//
// EPI 2 (LM head without a backward pass): the logits leave as three numbers a row and 64 columns - the largest logit z, the sum
// of exp((z - largest) / temperature) and the same sum weighted with z, of logits rounded to bf16 - which tgemm_stats_kernel
// merges: 1 / 11 of the bytes, and no pass that reads the logits again. 32768 x 151936 from 1536 deep: 11.45 ms with the logits
// and 1.68 for the pass over them, now 11.80 + 0.21. What the exponentials cost (two bf16 logits a conversion, one fma and one
// v_exp_f32 each, no subtraction: 11.98 -> 11.8) the other wave row waits for.
//
// GRP: the same product for rows sorted by expert, each expert's with its own B (routed experts). A row tile never straddles
// two experts; its tail rows repeat the expert's last one and are not stored.
template <int EPI, bool NN, bool GRP>
__global__ __launch_bounds__(512) void tgemm_kernel(const TGArgs a) {
  constexpr int TN = EPI == 1 ? 128 : 256;  // output columns per tile
  constexpr bool PARTS = EPI == 0 && !GRP;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wave >> 2, wc = wave & 3;

  // ---- tile sequence number -> output tile
  const tg_table_t table = (tg_table_t)a.table;
  const int tiles_m = GRP ? table[0].x : a.tiles_m;
  const int tiles = tiles_m * a.tiles_n, whole = PARTS ? a.whole : tiles;
  const int ntiles = PARTS ? whole + (tiles - whole) * a.splits : tiles;  // work items
  if (GRP && (int)blockIdx.x >= ntiles) return;  // (the grid is an upper bound)
  struct Tile {
    int m0, n0, k0, kt, mlim, e;  // origin; reduction from k0 on, K tiles; end of the rows; expert
    float* part;
  };
  auto tile_origin = [&](int id) __attribute__((always_inline)) {
    Tile t;
    const bool in_part = PARTS && id >= whole;
    const int base = in_part ? whole : 0, nb = in_part ? ntiles - whole : whole;
    const int q = nb >> 3, r = nb & 7, x = (id - base) & 7;
    int wg = base + (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + ((id - base) >> 3);
    t.k0 = 0;
    t.kt = a.K >> 6;
    t.part = nullptr;
    if (in_part) {  // part by part: what runs together on an XCD shares the reduction range
      const int rest = tiles - whole, split = (wg - whole) / rest;
      t.part = a.part + ((size_t)(wg - whole) << 16);
      wg -= split * rest;
      t.k0 = split * a.chunk * 128;
      t.kt = min(t.kt - split * a.chunk * 2, a.chunk * 2);
    }
    const int per_band = TG_GROUP_M * a.tiles_n;
    const int band = wg / per_band, first = band * TG_GROUP_M;
    const int rows = min(tiles_m - first, TG_GROUP_M);
    const int in_band = wg - band * per_band;
    t.n0 = (in_band / rows) * TN;
    const int mt = first + in_band % rows;
    if (GRP) {
      t.m0 = table[1 + mt].x;
      t.mlim = table[1 + mt].y;
      t.e = table[1 + mt].z;
    } else {
      t.m0 = mt * 256;
      t.mlim = a.M;
      t.e = 0;
    }
    return t;
  };

  // ---- staging: thread -> row (wave * 8 + lane / 8) of a 64-row issue, physical chunk lane & 7
  const int srow = wave * 8 + (lane >> 3);
  const int schunk = (lane & 7) ^ ((srow >> 1) & 7);  // logical chunk whose data lands at physical chunk lane & 7
  // NN: thread -> reduction row (wave * 4 + lane / 16) of a 32-row issue, physical chunk lane & 15 of its 256 bytes
  const int wrow = wave * 4 + (lane >> 4);
  const int wpc = ((lane & 15) ^ (((lane >> 4) << 2) | (wave & 3))) * 8;
  const size_t stepB = NN ? (size_t)64 * a.ldb : 64;  // elements of B from K tile to K tile
  // NN, which takes any number of rows: rows of A past the last one are out of a buffer's range and cost the CU's load path nothing
  // (repeating the last one instead: 2 rows from 28672 deep to 2048 columns 38 us, so 26). One descriptor per K tile; byte offsets
  // of 256 rows fit 32 bits.
  constexpr bool RANGE_A = NN && !GRP;
  const unsigned rowA = (unsigned)a.lda * 2, vA = srow * rowA + schunk * 16;
  const bf16_t* baseA = nullptr;
  unsigned rangeA = 0;
  const bf16_t* srcA[2][2];  // [piece][issue]
  const bf16_t* srcB[2][2];
  auto set_sources = [&](const Tile& t) __attribute__((always_inline)) {
    const int m0 = t.m0, n0 = t.n0, k0 = t.k0;
    const bf16_t* B = GRP ? a.B + t.e * a.stride : a.B;
    if (RANGE_A) {
      baseA = a.A + (size_t)m0 * a.lda + k0;
      rangeA = (unsigned)(min(a.M - m0, 256) - 1) * rowA + 128;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (!RANGE_A) {
          int row = m0 + i * 128 + h * 64 + srow;
          row = row < t.mlim ? row : t.mlim - 1;
          srcA[h][i] = a.A + (size_t)row * a.lda + schunk * 8 + (PARTS ? k0 : 0);
        }
        int col;
        if (NN) {  // one pointer: N is a multiple of 256 here, pieces and issues are a fixed step apart
          if (h == 0 && i == 0) srcB[0][0] = B + (size_t)(k0 + wrow) * a.ldb + n0 + (wpc >> 5) * 64 + (wpc & 31);
          continue;
        }
        if (EPI == 1) {  // piece h: gate (0) or up (1) rows of the tile's 128 columns, 32 per wave column
          col = n0 + (i * 2 + (wave >> 2)) * 32 + (wave & 3) * 8 + (lane >> 3);
          col = (col < a.N ? col : a.N - 1) + h * a.N;
        } else {
          col = n0 + (i * 2 + (wave >> 2)) * 64 + h * 32 + (wave & 3) * 8 + (lane >> 3);
          col = col < a.N ? col : a.N - 1;
        }
        srcB[h][i] = B + (size_t)col * a.ldb + schunk * 8 + (PARTS ? k0 : 0);
      }
  };
  auto stage = [&](int buf, int piece, int kt) __attribute__((always_inline)) {
    char* dst = smem + buf * TG_BUF + piece * TG_PIECE + wave * 1024;
    if (RANGE_A && piece < 2) {
      const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(baseA + (size_t)kt * 64), 0, rangeA, 0x00020000);
      const unsigned v = vA + piece * 64 * rowA;  // the whole offset in the vector operand, the one that the range check is about
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lptr_t)dst, 16, v, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lptr_t)(dst + 8192), 16, v + 128 * rowA, 0, 0, 0);
      return;
    }
    const bf16_t* s0 = piece < 2 ? srcA[piece][0] : NN ? srcB[0][0] + (piece - 2) * 32 : srcB[piece - 2][0];
    const bf16_t* s1 = piece < 2 ? srcA[piece][1] : NN ? s0 + stepB / 2 : srcB[piece - 2][1];
    const size_t at = kt * (piece < 2 ? (size_t)64 : stepB);
    __builtin_amdgcn_global_load_lds((gptr_t)(s0 + at), (lptr_t)dst, 16, 0, 0);
    __builtin_amdgcn_global_load_lds((gptr_t)(s1 + at), (lptr_t)(dst + 8192), 16, 0, 0);
  };

  // ---- fragment reads
  const int fr = lane & 15, fq = lane >> 4;
  const int sw = (fr >> 1) & 7;
  const int cb0 = ((fq) ^ sw) << 4, cb1 = ((4 + fq) ^ sw) << 4;
  const int a_off = (wr * 64 + fr) * 128, b_off = (wc * 32 + fr) * 128;
  bf16x8 af[4][2];
  tg_bfrag bf0, bf1;
  auto read_a = [&](int buf, int h) __attribute__((always_inline)) {
    const char* p = smem + buf * TG_BUF + h * TG_PIECE + a_off;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      af[mt][0] = *reinterpret_cast<const bf16x8*>(p + mt * 2048 + cb0);
      af[mt][1] = *reinterpret_cast<const bf16x8*>(p + mt * 2048 + cb1);
    }
  };
  // NN: pieces of [64 reduction rows][128 columns]; lane (fr, fq) needs rows 8 fq .. 8 fq + 7 of column fr, two transposed reads
  int t_adr[2][2];  // [16-column tile][row half]
#pragma unroll
  for (int nt = 0; nt < 2; ++nt)
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2)
      t_adr[nt][h2] = (int)(tr_addr((const char*)0, 8 * fq + 4 * h2, wc * 32 + nt * 16, fr) - (const char*)0);
  auto read_b = [&](int buf, int h, tg_bfrag& bf) __attribute__((always_inline)) {
    if (NN) {
      const uint32_t p = (uint32_t)(uintptr_t)(lptr_t)smem + buf * TG_BUF;
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int s = 0; s < 2; ++s)
          bf[nt][s] = cat4(tg_tr(p + t_adr[nt][0], (2 + h) * TG_PIECE + s * 8192), tg_tr(p + t_adr[nt][1], (2 + h) * TG_PIECE + s * 8192));
      return;
    }
    const char* p = smem + buf * TG_BUF + (2 + h) * TG_PIECE + b_off;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      bf[nt][0] = *reinterpret_cast<const bf16x8*>(p + nt * 2048 + cb0);
      bf[nt][1] = *reinterpret_cast<const bf16x8*>(p + nt * 2048 + cb1);
    }
  };
  tg_acc acc00, acc01, acc10, acc11;  // [m half][n half]
  auto mma = [&](tg_acc& acc, tg_bfrag& bf) __attribute__((always_inline)) {
    tg_barrier();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[nt][ks], af[mt][ks], acc[mt][nt], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    tg_barrier();
  };

  // ---- result stores. Lane (row fr, column quad fq) of tile (mt, nt) holds 4 consecutive columns; the two 16-column
  // tiles of a quadrant exchange halves between neighbouring 16-lane rows (v_permlane16_swap), after which a lane holds
  // 8 consecutive columns of one of them, 16-byte chunk out_ch of the quadrant's 64 bytes.
  const int out_ch = (fq & 1) * 2 + (fq >> 1);
  auto pack8 = [&](const f32x4& v0, const f32x4& v1) __attribute__((always_inline)) {
    unsigned pk[2][2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const f32x4& v = nt ? v1 : v0;
      bf16x2 lo = {f2bf(v[0]), f2bf(v[1])}, hi = {f2bf(v[2]), f2bf(v[3])};
      pk[nt][0] = __builtin_bit_cast(unsigned, lo);
      pk[nt][1] = __builtin_bit_cast(unsigned, hi);
    }
    const auto r0 = __builtin_amdgcn_permlane16_swap(pk[0][0], pk[1][0], false, false);
    const auto r1 = __builtin_amdgcn_permlane16_swap(pk[0][1], pk[1][1], false, false);
    return u32x4{r0[0], r1[0], r0[1], r1[1]};
  };
  Tile cur = {};  // the output tile being computed
  auto store8 = [&](auto stream, int m, int n, u32x4 o) __attribute__((always_inline)) {
    if (m < cur.mlim && n < a.N) {
      bf16_t* p = a.C + (size_t)m * a.ldc + n;
      if (n + 8 <= a.N) {
        if constexpr (decltype(stream)::value)
          __builtin_nontemporal_store(o, reinterpret_cast<u32x4*>(p));
        else
          *reinterpret_cast<u32x4*>(p) = o;
      } else {  // the last 4 columns of a width that is not a multiple of 8
        *reinterpret_cast<u32x2*>(p) = (u32x2){o[0], o[1]};
      }
    }
  };
  // plain form: both column quadrants of a row half, 32 rows of 128 bytes at a time through the wave's 4 KiB
  auto put = [&](tg_acc& c0, tg_acc& c1, int mh) __attribute__((always_inline)) {
    const int m0 = cur.m0, n0 = cur.n0;
    float* part = cur.part;
    char* ob = smem + TG_LDS + wave * 4096;
    if (PARTS && part) {  // one part of the reduction, summed by a kernel of its own
      float* op = part + (wr * 128 + mh * 64 + fr) * 256 + wc * 64 + fq * 4;
      const int left = a.M - m0 - wr * 128 - mh * 64 - fr;  // rows past the last one are not read (2 rows, 28 parts: 58 MB of them)
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
        if (mt * 16 < left)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
          *reinterpret_cast<f32x4*>(op + mt * 4096 + nt * 16) = c0[mt][nt];
          *reinterpret_cast<f32x4*>(op + mt * 4096 + 32 + nt * 16) = c1[mt][nt];
        }
      return;
    }
    if (!NN && !GRP && a.bias) {
#pragma unroll
      for (int nh = 0; nh < 2; ++nh)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
          const int nb = n0 + wc * 64 + nh * 32 + nt * 16 + fq * 4;
          if (nb < a.N) {
            const bf16x4 bb = *reinterpret_cast<const bf16x4*>(a.bias + nb);
#pragma unroll
            for (int mt = 0; mt < 4; ++mt)
#pragma unroll
              for (int j = 0; j < 4; ++j) (nh ? c1 : c0)[mt][nt][j] += bf2f(bb[j]);
          }
        }
    }
#pragma unroll
    for (int hb = 0; hb < 2; ++hb) {
#pragma unroll
      for (int mi = 0; mi < 2; ++mi) {
        const int mt = hb * 2 + mi;
        char* row = ob + (mi * 16 + fr) * 128;
        *reinterpret_cast<u32x4*>(row + ((out_ch ^ (fr & 7)) << 4)) = pack8(c0[mt][0], c0[mt][1]);
        *reinterpret_cast<u32x4*>(row + (((out_ch + 4) ^ (fr & 7)) << 4)) = pack8(c1[mt][0], c1[mt][1]);
      }
      u32x4 o[4];
      const int r8 = lane >> 3, ch = lane & 7;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = *reinterpret_cast<const u32x4*>(ob + (i * 8 + r8) * 128 + ((ch ^ r8) << 4));
#pragma unroll
      for (int i = 0; i < 4; ++i) store8(std::true_type{}, m0 + wr * 128 + mh * 64 + hb * 32 + i * 8 + r8, n0 + wc * 64 + ch * 8, o[i]);
    }
  };
  // gated form: `g` and `u` are the two column quadrants of one row half. A wave's 32 result columns are half a line: the four
  // waves of a wave row passing them on together through LDS was slower (1361 against 1321 us at 32768 x 8960 from 1536 deep)
  // than storing from the registers; so was dealing the activation out over the next tile's first phases (1333).
  auto put_gated = [&](tg_acc& g, tg_acc& u, int mh) __attribute__((always_inline)) {
    const int m0 = cur.m0, n0 = cur.n0;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      f32x4 v[2];
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // the unfused path carries gate|up as a bf16 tensor
          const float gg = bf2f(f2bf(g[mt][nt][j])), uu = bf2f(f2bf(u[mt][nt][j]));
          v[nt][j] = tg_silu(gg) * uu;
        }
      store8(std::false_type{}, m0 + wr * 128 + mh * 64 + mt * 16 + fr, n0 + wc * 32 + out_ch * 8, pack8(v[0], v[1]));
    }
  };

  // statistics: a wave's 64 columns of a row half. The four 16-lane rows hold 4 of every 16 columns of the same 16 result rows.
  auto put_stats = [&](tg_acc& c0, tg_acc& c1, int mh) __attribute__((always_inline)) {
    const int col = cur.n0 + wc * 64;
    if (col >= a.N) return;
    const bool edge = col + 64 > a.N;  // columns behind the last one (whole quads) repeat it in the operands: left out
    float keep[3] = {0.f, 0.f, 0.f};   // row mt = fq of this lane's four
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      float mx = -INFINITY, sum = 0.f, ws = 0.f;
      float z[2][2][4];
#pragma unroll
      for (int nh = 0; nh < 2; ++nh)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
          const f32x4& v = (nh ? c1 : c0)[mt][nt];
#pragma unroll
          for (int j = 0; j < 4; j += 2) {
            const bf16x2 p = {f2bf(v[j]), f2bf(v[j + 1])};
            const unsigned u = __builtin_bit_cast(unsigned, p);
            z[nh][nt][j] = __uint_as_float(u << 16);
            z[nh][nt][j + 1] = __uint_as_float(u & 0xffff0000u);
          }
          if (edge && col + nh * 32 + nt * 16 + fq * 4 >= a.N) continue;
#pragma unroll
          for (int j = 0; j < 4; ++j) mx = fmaxf(mx, z[nh][nt][j]);
        }
      mx = max_xor16(max_xor32(mx));
      // rounded: the merge takes the difference back. A block of nothing but -inf (forbidden ids) adds nothing to the row's sum
      const float ref = mx > -INFINITY ? mx * a.scale : 0.f;
#pragma unroll
      for (int nh = 0; nh < 2; ++nh)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
          if (edge && col + nh * 32 + nt * 16 + fq * 4 >= a.N) continue;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float e = __builtin_amdgcn_exp2f(fmaf(z[nh][nt][j], a.scale, -ref));
            sum += e;
            ws = fmaf(e, z[nh][nt][j], ws);
          }
        }
      sum = sum_xor16(sum_xor32(sum));
      ws = sum_xor16(sum_xor32(ws));
      if (fq == mt) {
        keep[0] = mx;
        keep[1] = sum;
        keep[2] = ws;
      }
    }
    const int m = cur.m0 + wr * 128 + mh * 64 + lane;  // = .. + fq * 16 + fr
    if (m < a.M) {
      const size_t cbs = (a.N + 63) >> 6;
      float* op = a.part + (size_t)(col >> 6) * a.M + m;
#pragma unroll
      for (int i = 0; i < 3; ++i) op[i * cbs * a.M] = keep[i];
    }
  };

  // One K tile = four phases. The K tiles of the block's successive output tiles form ONE stream: the pieces staged
  // while the last two K tiles of an output tile are computed are K tiles 0 and 1 of the NEXT output tile, so the
  // prologue's load latency is paid once per block and the result stores run under the next tile's loads.
  // MODE 0: inside an output tile (K tiles t+1, t+2 belong to it). MODE 1: second to last K tile (t+1 is the last one;
  // "t+2" is K tile 0 of the next output tile, whose source addresses replace the current ones after phase 1).
  // MODE 2: last K tile ("t+1", "t+2" are K tiles 0, 1 of the next output tile). Without a next tile nothing is staged
  // and the loads still in flight are drained.
  Tile next = {};
  bool has_next = false;
  auto tile = [&](auto buf_c, int t, auto mode_c) __attribute__((always_inline)) {
    constexpr int buf = decltype(buf_c)::value, MODE = decltype(mode_c)::value;
    const bool go = MODE == 0 || has_next;
    const int t1 = MODE == 2 ? 0 : t + 1, t2 = MODE == 0 ? t + 2 : MODE - 1;
    // phase 1: quadrant (0, 0)
    read_b(buf, 0, bf0);
    __builtin_amdgcn_sched_barrier(0);
    read_a(buf, 0);
    if (MODE < 2 || go) stage(buf ^ 1, PA1, t1);
    // the four B0 reads (issued first) have returned before this phase's first barrier: B0 is restaged one phase
    // from now, when the staggered wave group has only just passed that barrier
    asm volatile("s_waitcnt lgkmcnt(8)" ::: "memory");
    mma(acc00, bf0);
    if (MODE == 1 && go) set_sources(next);
    // phase 2: quadrant (0, 1)
    read_b(buf, 1, bf1);
    if (go) stage(buf, PB0, t2);
    mma(acc01, bf1);
    // last K tile: a row half is final once its phases are over; it leaves while the other wave group computes
    if (MODE == 2 && EPI == 0) put(acc00, acc01, 0);
    if (MODE == 2 && EPI == 1) put_gated(acc00, acc01, 0);
    if (MODE == 2 && EPI == 2) put_stats(acc00, acc01, 0);
    // phase 3: quadrant (1, 1)
    read_a(buf, 1);
    if (go) stage(buf, PA0, t2);
    mma(acc11, bf1);
    // phase 4: quadrant (1, 0); the next K tile of the stream becomes readable
    if (go) {
      stage(buf, PB1, t2);
      tg_vmcnt<6>();
    } else if (MODE == 1) {
      tg_vmcnt<0>();
    }
    mma(acc10, bf0);
    if (MODE == 2 && EPI == 0) put(acc10, acc11, 1);
    if (MODE == 2 && EPI == 1) put_gated(acc10, acc11, 1);
    if (MODE == 2 && EPI == 2) put_stats(acc10, acc11, 1);
  };
  using B0 = std::integral_constant<int, 0>;
  using B1 = std::integral_constant<int, 1>;
  using M0 = std::integral_constant<int, 0>;
  using M1 = std::integral_constant<int, 1>;
  using M2 = std::integral_constant<int, 2>;

  // ---- prologue: K tile 0 whole, B0 A0 B1 of K tile 1 (its A1 leaves in phase 1 of K tile 0)
  int id = blockIdx.x;
  cur = tile_origin(id);
  set_sources(cur);
  stage(0, PB0, 0);
  stage(0, PA0, 0);
  stage(0, PB1, 0);
  stage(0, PA1, 0);
  stage(1, PB0, 1);
  stage(1, PA0, 1);
  stage(1, PB1, 1);
  tg_vmcnt<6>();
  tg_barrier();
  if (wr == 1) tg_barrier();  // the second wave row runs one barrier behind

  while (true) {
    const int nid = id + gridDim.x;
    has_next = nid < ntiles;
    if (has_next) next = tile_origin(nid);
    const int KT = cur.kt;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        acc00[mt][nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
        acc01[mt][nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
        acc10[mt][nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
        acc11[mt][nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
      }
    // K tiles come in pairs (K is a multiple of 128)
    int t = 0;
    for (; t + 2 < KT; t += 2) {
      tile(B0{}, t, M0{});
      tile(B1{}, t + 1, M0{});
    }
    tile(B0{}, t, M1{});
    tile(B1{}, t + 1, M2{});
    if (!has_next) break;
    id = nid;
    cur = next;
  }
  if (wr == 0) tg_barrier();
}

// Row tiles of 256 of the experts' rows (offsets [E + 1]), in order: table[0].x = their number, then {first row, end of the
// expert's rows, expert} each. One block.
__global__ __launch_bounds__(256) void tgemm_table_kernel(const int* __restrict__ offsets, int E, int4* __restrict__ table) {
  __shared__ int wsum[4];
  const int t = threadIdx.x, lane = t & 63;
  int base = 0;
  for (int e0 = 0; e0 < E; e0 += 256) {
    const int e = e0 + t;
    const int lo = e < E ? offsets[e] : 0, hi = e < E ? offsets[e + 1] : 0, n = (hi - lo + 255) / 256;
    int incl = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(incl, o, 64);
      if (lane >= o) incl += y;
    }
    if (lane == 63) wsum[t >> 6] = incl;
    __syncthreads();
    int at = base + incl - n;
    for (int w = 0; w < 4; ++w) {
      if (w < (t >> 6)) at += wsum[w];
      base += wsum[w];
    }
    __syncthreads();
    for (int i = 0; i < n; ++i) table[1 + at + i] = make_int4(lo + i * 256, hi, e, 0);
  }
  if (t == 0) table[0] = make_int4(base, 0, 0, 0);
}

// =====================================================================================
// Weight gradient:  dW[N, K] (fp32) += dY[M, N]^T . X[M, K]     (bf16 operands, both token-major)
//
// The same phase structure as above with the roles  rows -> n (columns of dY), columns -> k (columns of X), reduction
// -> tokens. Both operands are stored with the REDUCTION index as the slow dimension, so the staged pieces are
// token-major [64 tokens][128 columns] (256-byte rows, the swizzle of flash_tiles.hpp) and every MFMA operand is a pair
// of transposed LDS reads (ds_read_b64_tr_b16: a lane receives 4 consecutive tokens of one column; 8 rows of 32 bytes for
// 32 lanes, which the swizzle puts on different banks).
//   A0 / A1 = dY columns [0, 64) / [64, 128) of both wave rows; B0 / B1 = X columns [0, 32) / [32, 64) of all four
//   wave columns - as for the forward kernel, pieces are what one phase reads.
// 16x16x32 products, not 32x32x16: where all CUs are busy 5 % faster (17920 x 1536 over 32768 tokens: 1481 -> 1407 us); where half of
// them idle up to 5 % slower, for twice the transposed reads of A (2560 x 2560 over 2000 tokens, 100 tiles: 45 -> 48).
// A tile whose whole reduction falls to one workgroup is added with a plain read-add-write. The tiles that would leave CUs
// idle in a last round are reduced by several workgroups, `chunk` 128-token pairs each, that write their sums as fp32 to
// `part`; tgemm_wgrad_sum_kernel adds them. fp32 atomics on the gradient instead execute at the memory side, 1.3 TB/s
// chip-wide, in any order; over 32768 tokens, us with atomics / with parts: 1536 x 1536 171 / 140, 2048 x 1536 197 / 184,
// 17920 x 1536 1450 / 1412; over 16384: 2048 x 4096 263 / 225, 5120 x 2048 347 / 316.
// =====================================================================================
struct TWArgs {
  const bf16_t* dY;
  long ldy;
  const bf16_t* X;
  long ldx;
  float* dW;
  long ldw;
  int M, N, K;
  int tiles_n, tiles_k;
  int pairs;          // 128-token pairs of K tiles in M, the last one possibly ragged
  int whole;          // the first `whole` tiles are reduced by one workgroup each
  int splits, chunk;  // the others: workgroups per tile, pairs per workgroup (the last one of a tile may get fewer)
  float* part;        // [tile - whole][splits][wave][m half][n half][mt][nt][lane][4]
  // grouped (GRP): rows offsets[e] .. offsets[e + 1] belong to expert e, whose gradient lies `stride` elements from the last
  const int* offsets;
  long stride;
  int band = 8;  // tgemm_wgrad_few_kernel: tile rows that are walked together
};

typedef f32x4 __attribute__((aligned(4))) f32x4u;
constexpr long TG_STREAM = 1l << 26;  // elements of an fp32 gradient that the memory-side cache cannot hold

DEVINL void tg_wgrad_origin(const TWArgs& a, int wg, int& n0, int& k0) {
  const int per_band = TG_GROUP_M * a.tiles_k;
  const int band = wg / per_band, first = band * TG_GROUP_M;
  const int rows = min(a.tiles_n - first, TG_GROUP_M);
  const int in_band = wg - band * per_band;
  n0 = (first + in_band % rows) * 256;
  k0 = (in_band / rows) * 256;
}

// NT: a gradient larger than the 256 MB of the memory-side cache is streamed past the caches (us, 151936 x 1536, 1024 / 2048 / 4096 / 16384
// tokens 637 / 594, 949 / 925, 1662 / 1605, 5726 / 5728; 128 experts of 1536 x 2048, 1024 rows each 1131 / 1076). A smaller one may be
// there still, from its clearing or the last pass: 17920 x 1536, 1024 tokens 74 us, streamed 86.
template <bool GRP, bool NT>
__global__ __launch_bounds__(512) void tgemm_wgrad_kernel(const TWArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wave >> 2, wc = wave & 3;

  // ---- this workgroup's range of work units (tile, pair): `chunk` pairs of one tile. Ids are dealt round-robin to
  // the 8 XCDs: the workgroups of one XCD take neighbouring tiles, which share dY / X panels in its L2.
  // (whole tiles and split tiles are renumbered separately: the hardware starts workgroups in id order, and the long
  // whole-tile workgroups have to start first; `whole` is 0, a multiple of 256, or the whole grid)
  const bool in_whole = GRP || (int)blockIdx.x < a.whole;
  const int base = in_whole ? 0 : a.whole, nb = in_whole ? a.whole : (int)gridDim.x - a.whole;
  const int id = blockIdx.x - base;
  const int xq = nb >> 3, xr = nb & 7, xx = id & 7;
  const int b = base + (xx < xr ? xx * (xq + 1) : xr * (xq + 1) + (xx - xr) * xq) + (id >> 3);
  int b_tile = b, b_split = 0, b_chunk = a.pairs, row_lo = 0, row_hi = a.M;
  float* dW = a.dW;
  if (GRP) {
    const int per = a.tiles_n * a.tiles_k, e = b / per;
    b_tile = b - e * per;
    row_lo = a.offsets[e];
    row_hi = a.offsets[e + 1];
    if (row_hi <= row_lo) return;  // an expert without rows adds nothing
    dW += e * a.stride;
    b_chunk = (row_hi - row_lo + 127) / 128;
  } else if (b >= a.whole) {
    b_tile = a.whole + (b - a.whole) / a.splits;
    b_split = (b - a.whole) - (b_tile - a.whole) * a.splits;
    b_chunk = a.chunk;
  }
  // ---- staging: thread -> token row (wave * 4 + lane / 16) of a 32-row issue, physical 16-byte chunk lane & 15
  const int srow = wave * 4 + (lane >> 4);
  const int pc = ((lane & 15) ^ (((lane >> 4) << 2) | (wave & 3))) * 8;  // piece column whose chunk lands here
  // Rows past the last token are out of the buffer's range: such loads write zeros. One descriptor per piece and K tile
  // (scalar registers), of no more than 64 rows: byte offsets stay small however large the operand is.
  const bf16_t *pA = nullptr, *pB = nullptr;  // the segment's first token, column n0 / k0
  unsigned vA = 0, vB = 0;                    // this lane's byte offset of a piece's first row and column
  int tokens = 0;                             // of the segment
  auto stage = [&](int buf, int piece, int kt) __attribute__((always_inline)) {
    char* dst = smem + buf * TG_BUF + piece * TG_PIECE + wave * 1024;
    const bool isA = piece < 2;
    const unsigned row = (unsigned)(isA ? a.ldy : a.ldx) * 2;  // bytes
    const int rows = min(tokens - kt * 64, 64);
    const unsigned range = rows > 0 ? (rows - 1) * row + min(row, 512u) : 0u;
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>((isA ? pA : pB) + (size_t)kt * 32 * row), 0, range, 0x00020000);
    // the whole offset in the vector operand, the one that the range check is about
    const unsigned v = (isA ? vA : vB) + (piece & 1) * (isA ? 128 : 64);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lptr_t)dst, 16, v, 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lptr_t)(dst + 8192), 16, v + 32 * row, 0, 0, 0);
  };

  // ---- transposed fragment reads: addresses inside a piece (the same for both buffers and every 32-token slab). Lane (fr, fq)
  // of an operand holds tokens 8 fq .. 8 fq + 7 of column fr: two reads of four tokens
  const int fr = lane & 15, fq = lane >> 4;
  int a_adr[4][2], b_adr[2][2];  // [16-column tile][token half]
#pragma unroll
  for (int h2 = 0; h2 < 2; ++h2) {
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
      a_adr[mt][h2] = (int)(tr_addr((const char*)0, 8 * fq + 4 * h2, wr * 64 + mt * 16, fr) - (const char*)0);
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
      b_adr[nt][h2] = (int)(tr_addr((const char*)0, 8 * fq + 4 * h2, wc * 32 + nt * 16, fr) - (const char*)0);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lptr_t)smem;
  bf16x8 af[4][2];  // [16-column tile][32-token slab]
  tg_bfrag bf0, bf1;
  auto read_a = [&](int buf, int h) __attribute__((always_inline)) {
    const uint32_t p = lds0 + buf * TG_BUF;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int s = 0; s < 2; ++s)
        af[mt][s] = cat4(tg_tr(p + a_adr[mt][0], h * TG_PIECE + s * 8192), tg_tr(p + a_adr[mt][1], h * TG_PIECE + s * 8192));
  };
  auto read_b = [&](int buf, int h, tg_bfrag& bf) __attribute__((always_inline)) {
    const uint32_t p = lds0 + buf * TG_BUF;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int s = 0; s < 2; ++s)
        bf[nt][s] = cat4(tg_tr(p + b_adr[nt][0], (2 + h) * TG_PIECE + s * 8192), tg_tr(p + b_adr[nt][1], (2 + h) * TG_PIECE + s * 8192));
  };
  tg_acc acc00, acc01, acc10, acc11;  // [n half][k half]
  auto mma = [&](tg_acc& acc, tg_bfrag& bf) __attribute__((always_inline)) {
    tg_barrier();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[nt][s], af[mt][s], acc[mt][nt], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    tg_barrier();
  };
  // TAIL 0: tiles t+1 and t+2 exist; 1: only t+1 exists; 2: last tile
  auto tile = [&](auto buf_c, int t, auto tail_c) __attribute__((always_inline)) {
    constexpr int buf = decltype(buf_c)::value, TAIL = decltype(tail_c)::value;
    read_b(buf, 0, bf0);
    __builtin_amdgcn_sched_barrier(0);
    read_a(buf, 0);
    if (TAIL < 2) stage(buf ^ 1, PA1, t + 1);
    asm volatile("s_waitcnt lgkmcnt(15)" ::: "memory");  // the eight B0 reads, issued first of 24, have returned (see the forward kernel; the counter holds at most 15)
    mma(acc00, bf0);
    read_b(buf, 1, bf1);
    if (TAIL < 1) stage(buf, PB0, t + 2);
    mma(acc01, bf1);
    read_a(buf, 1);
    if (TAIL < 1) stage(buf, PA0, t + 2);
    mma(acc11, bf1);
    if (TAIL < 1) stage(buf, PB1, t + 2);
    if (TAIL == 0) tg_vmcnt<6>();
    if (TAIL == 1) tg_vmcnt<0>();
    mma(acc10, bf0);
  };
  using B0 = std::integral_constant<int, 0>;
  using B1 = std::integral_constant<int, 1>;
  using T0 = std::integral_constant<int, 0>;
  using T1 = std::integral_constant<int, 1>;
  using T2 = std::integral_constant<int, 2>;

  // ---- one segment: pairs [p0, p1) of one output tile
  int n0, k0;
  const int p0 = b_split * b_chunk, p1 = GRP ? b_chunk : min(a.pairs, p0 + b_chunk);
  tg_wgrad_origin(a, b_tile, n0, k0);
  const int tok0 = row_lo + p0 * 128, KT = (p1 - p0) * 2;
  tokens = row_hi - tok0;
  // N may end half way through the last tile row (N % 256 == 128): the second wave row then re-reads the first
  // one's columns and does not write
  const bool half_n = n0 + 128 >= a.N;
  pA = a.dY + (size_t)tok0 * a.ldy + n0;
  pB = a.X + (size_t)tok0 * a.ldx + k0;
  vA = (unsigned)(srow * a.ldy + (half_n ? 0 : (pc >> 6) * 128) + (pc & 63)) * 2;
  vB = (unsigned)(srow * a.ldx + (pc >> 5) * 64 + (pc & 31)) * 2;
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      acc00[mt][nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
      acc01[mt][nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
      acc10[mt][nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
      acc11[mt][nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
  stage(0, PB0, 0);
  stage(0, PA0, 0);
  stage(0, PB1, 0);
  stage(0, PA1, 0);
  stage(1, PB0, 1);
  stage(1, PA0, 1);
  stage(1, PB1, 1);
  tg_vmcnt<6>();
  tg_barrier();
  if (wr == 1) tg_barrier();  // the second wave row runs one barrier behind
  int t = 0;
  for (; t + 2 < KT; t += 2) {
    tile(B0{}, t, T0{});
    tile(B1{}, t + 1, T0{});
  }
  tile(B0{}, t, T1{});
  tile(B1{}, t + 1, T2{});
  if (wr == 0) tg_barrier();  // from here on nobody reads a staged tile: a wave has 16 KiB of LDS to itself

  // ---- lane (row fr, fq) of tile (mt, nt) holds 4 consecutive k columns
  if (half_n && wr == 1) return;
  if (!GRP && b >= a.whole) {
    f32x4* pp = reinterpret_cast<f32x4*>(a.part + ((size_t)(b - a.whole) << 16)) + wave * 2048 + lane;
    auto put = [&](tg_acc& acc, int q) __attribute__((always_inline)) {
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) pp[(q * 8 + mt * 2 + nt) * 64] = acc[mt][nt];
    };
    put(acc00, 0);
    put(acc01, 1);
    put(acc10, 2);
    put(acc11, 3);
    return;
  }
  // a row half (64 x 64 fp32) passes through the wave's LDS: an instruction then moves 256 bytes of four rows
  char* ob = smem + wave * 16384;
  auto flush = [&](tg_acc& c0, tg_acc& c1, int mh) __attribute__((always_inline)) {
    float* op = dW + (size_t)(n0 + wr * 128 + mh * 64) * a.ldw + k0 + wc * 64;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int nh = 0; nh < 2; ++nh)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          *reinterpret_cast<f32x4*>(ob + (mt * 16 + fr) * 256 + (((nh * 8 + nt * 4 + fq) ^ fr) << 4)) = (nh ? c1 : c0)[mt][nt];
#pragma unroll
    for (int i0 = 0; i0 < 16; i0 += 8) {
      f32x4 old[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const f32x4u* p = reinterpret_cast<const f32x4u*>(op + (size_t)((i0 + i) * 4 + fq) * a.ldw + fr * 4);
        if constexpr (NT)
          old[i] = __builtin_nontemporal_load(p);
        else
          old[i] = *p;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int row = (i0 + i) * 4 + fq;
        const f32x4 v = *reinterpret_cast<const f32x4*>(ob + row * 256 + ((fr ^ (row & 15)) << 4));
        f32x4u* p = reinterpret_cast<f32x4u*>(op + (size_t)row * a.ldw + fr * 4);
        if constexpr (NT)
          __builtin_nontemporal_store(old[i] + v, p);
        else
          *p = old[i] + v;
      }
    }
  };
  flush(acc00, acc01, 0);
  flush(acc10, acc11, 1);
}

// dW += the parts of the tiles from `whole` on, in order. Block: 32 rows x 64 columns of a tile (a wave's quarter of a row
// half); a thread has 4 columns of 2 of the rows, 8 threads a 128-byte line.
__global__ __launch_bounds__(256) void tgemm_wgrad_sum_kernel(const TWArgs a) {
  const int t = blockIdx.x >> 5, wave = (blockIdx.x >> 2) & 7, mh = (blockIdx.x >> 1) & 1, mt2 = blockIdx.x & 1;
  int n0, k0;
  tg_wgrad_origin(a, a.whole + t, n0, k0);
  const int fq = threadIdx.x & 3, nt = (threadIdx.x >> 2) & 1, nh = (threadIdx.x >> 3) & 1, fr = threadIdx.x >> 4;
  if (n0 + (wave >> 2) * 128 >= a.N) return;
  const f32x4* p = reinterpret_cast<const f32x4*>(a.part + ((size_t)t * a.splits << 16)) + wave * 2048 +
                   ((mh * 2 + nh) * 8 + mt2 * 4 + nt) * 64 + fq * 16 + fr;
  float* op = a.dW + (size_t)(n0 + (wave >> 2) * 128 + mh * 64 + mt2 * 32 + fr) * a.ldw + k0 + (wave & 3) * 64 + nh * 32 + nt * 16 + fq * 4;
  f32x4u* o0 = reinterpret_cast<f32x4u*>(op);
  f32x4u* o1 = reinterpret_cast<f32x4u*>(op + 16 * a.ldw);
  f32x4 v0 = p[0], v1 = p[128];
  const f32x4 d0 = *o0, d1 = *o1;
#pragma unroll 4
  for (int s = 1; s < a.splits; ++s) {
    v0 += p[(size_t)s << 14];
    v1 += p[((size_t)s << 14) + 128];
  }
  *o0 = d0 + v0;
  *o1 = d1 + v1;
}

// =====================================================================================
// Weight gradient over few tokens: tiles of 128 x 128, a workgroup of 4 waves (2 x 2, 64 x 64 each), three or four of them on a CU.
//
// Over few tokens the fp32 gradient is what moves: it is read and written once, 5 to 50 times the operands' bytes. The kernel above has
// one workgroup a CU, whose gradient passes behind its products, not beside them, and few tiles need parts and a second launch. Here
// one workgroup's products run beside another's gradient. A ring of S stages of 32 tokens, one barrier a stage; the gradient is
// streamed past the L2 (nontemporal: nothing reads it again soon, and the operands' panels stay there). What bounds it: the
// memory up to some 700 tokens, above that the LDS (32 KiB read and 16 KiB written a stage for 256 cycles of products: 6 us a tile
// and 1024 tokens with the CU full). us, gradient not in the caches, kernel above / this one: 17920 x 1536, 256 / 700 / 1500 tokens
// 59 / 48, 78 / 61, 107 / 93; 2048 x 1536 19 / 9.3, 28 / 14, 31 / 22; 151936 x 1536 425 / 340, 572 / 436, 789 / 798. Without
// streaming 700 tokens take 68, 15 and 514 us. S: 2 stages leave room for four workgroups, 3 for three, better where there are no
// more than three a CU (2048 x 1536, 1500 tokens 26 / 22; 22016 x 4096, 700 tokens 164 / 175; 4 stages 206).
// Sums are taken over all tokens in their order, as in a whole tile above and bit for bit as there; tiles that are split there stay
// there (1500 tokens of 2048 x 1536), for parts sum in shorter chains.
//
// GRP: routed experts' gradients, rows sorted by expert. us, 128 experts of 1536 x 2048, 64 / 256 / 512 / 700 rows an expert, kernel
// above / this one: 618 / 550, 710 / 561, 862 / 746, 992 / 871.
// =====================================================================================
constexpr int TWF_STAGE = 16 * 1024;  // 32 tokens x 128 columns of both operands

template <bool GRP, int S>
__global__ __launch_bounds__(256, S == 2 ? 4 : 3) void tgemm_wgrad_few_kernel(const TWArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wave >> 1, wc = wave & 1, fr = lane & 15, fq = lane >> 4;

  // ---- id -> tile: contiguous ranges per XCD, walked in bands of tile rows. Ranges of all experts' tiles (an expert's operands then
  // pass through one L2), or, where an expert alone has many, of each expert's: a crowded expert would keep one XCD busy
  int nb = gridDim.x, id = blockIdx.x, e = 0;
  if (GRP && a.chunk) {
    nb = a.tiles_n * a.tiles_k;
    e = id / nb;
    id -= e * nb;
  }
  const int xq = nb >> 3, xr = nb & 7, xx = id & 7;
  int b = (xx < xr ? xx * (xq + 1) : xr * (xq + 1) + (xx - xr) * xq) + (id >> 3);
  int row_lo = 0, row_hi = a.M;
  float* dW = a.dW;
  if (GRP) {
    if (!a.chunk) {
      const int per = a.tiles_n * a.tiles_k;
      e = b / per;
      b -= e * per;
    }
    row_lo = a.offsets[e];
    row_hi = a.offsets[e + 1];
    if (row_hi <= row_lo) return;  // an expert without rows adds nothing
    dW += e * a.stride;
  }
  const int per_band = a.band * a.tiles_k, band = b / per_band, in_band = b - band * per_band;
  const int band_rows = min(a.tiles_n - band * a.band, a.band);
  const int n0 = (band * a.band + in_band % band_rows) * 128, k0 = in_band / band_rows * 128;

  // ---- staging: thread -> token row (wave * 4 + lane / 16) of a 16-row issue; rows past the last token are out of the buffer's
  // range and write zeros (as in tgemm_wgrad_kernel)
  const int srow = wave * 4 + fq, pc = (fr ^ ((fq << 2) | wave)) * 8;
  const int tokens = row_hi - row_lo;
  const bf16_t* pA = a.dY + (size_t)row_lo * a.ldy + n0;
  const bf16_t* pB = a.X + (size_t)row_lo * a.ldx + k0;
  const unsigned rowA = (unsigned)a.ldy * 2, rowB = (unsigned)a.ldx * 2;  // bytes
  const unsigned vA = srow * rowA + pc * 2, vB = srow * rowB + pc * 2;
  auto stage = [&](int slot, int t) __attribute__((always_inline)) {
    char* dst = smem + slot * TWF_STAGE + wave * 1024;
    const int rows = min(tokens - t * 32, 32);
    const unsigned ra = rows > 0 ? (rows - 1) * rowA + 256 : 0u, rb = rows > 0 ? (rows - 1) * rowB + 256 : 0u;
    const auto sa = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(pA + (size_t)t * 16 * rowA), 0, ra, 0x00020000);
    const auto sb = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(pB + (size_t)t * 16 * rowB), 0, rb, 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(sa, (lptr_t)dst, 16, vA, 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(sa, (lptr_t)(dst + 4096), 16, vA + 16 * rowA, 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(sb, (lptr_t)(dst + 8192), 16, vB, 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(sb, (lptr_t)(dst + 12288), 16, vB + 16 * rowB, 0, 0, 0);
  };

  int a_adr[4][2], b_adr[4][2];  // [16-column tile][token half]
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) {
      a_adr[i][h2] = (int)(tr_addr((const char*)0, 8 * fq + 4 * h2, wr * 64 + i * 16, fr) - (const char*)0);
      b_adr[i][h2] = (int)(tr_addr((const char*)0, 8 * fq + 4 * h2, wc * 64 + i * 16, fr) - (const char*)0);
    }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lptr_t)smem;
  f32x4 acc[4][4] = {};  // [n tile][k tile]

  const int KT = (tokens + 31) >> 5;
#pragma unroll
  for (int i = 0; i < S - 1; ++i) stage(i, i);
  int slot = 0;
  for (int t = 0; t < KT; ++t) {
    tg_vmcnt<4 * (S - 2)>();
    tg_barrier();  // stage t is complete; everyone has read stage t - 1, which the next request overwrites
    const int next = slot == 0 ? S - 1 : slot - 1;
    stage(next, t + S - 1);
    const uint32_t p = lds0 + slot * TWF_STAGE;
    bf16x8 af[4], bf[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) bf[i] = cat4(tg_tr(p + b_adr[i][0], 8192), tg_tr(p + b_adr[i][1], 8192));
#pragma unroll
    for (int i = 0; i < 4; ++i) af[i] = cat4(tg_tr(p + a_adr[i][0], 0), tg_tr(p + a_adr[i][1], 0));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[nt], af[mt], acc[mt][nt], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    slot = slot == S - 1 ? 0 : slot + 1;
  }
  tg_vmcnt<0>();

  // ---- lane (fr, fq) of tile (mt, nt) holds 4 consecutive k columns of row fr; 32 rows at a time pass through 8 KiB of LDS, after
  // which an instruction moves 256 bytes of four rows
  float* op = dW + (size_t)(n0 + wr * 64 + fq) * a.ldw + k0 + wc * 64 + fr * 4;
  f32x4 old[16];
  auto fetch = [&](int i0, int i1) __attribute__((always_inline)) {
#pragma unroll
    for (int i = i0; i < i1; ++i) old[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4u*>(op + (size_t)i * 4 * a.ldw));
  };
  fetch(0, S == 2 ? 8 : 16);  // (four workgroups a CU: 128 registers)
  tg_barrier();               // from here on nobody reads a stage
  char* ob = smem + wave * 8192;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (S == 2 && h == 1) fetch(8, 16);
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) *reinterpret_cast<f32x4*>(ob + (m * 16 + fr) * 256 + (((nt * 4 + fq) ^ fr) << 4)) = acc[h * 2 + m][nt];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = i * 4 + fq;
      const f32x4 v = *reinterpret_cast<const f32x4*>(ob + row * 256 + ((fr ^ (row & 15)) << 4));
      __builtin_nontemporal_store(old[h * 8 + i] + v, reinterpret_cast<f32x4u*>(op + (size_t)(h * 8 + i) * 4 * a.ldw));
    }
  }
}

// =====================================================================================
// Input gradient:  dX[M, C] = dY[M, R] . W[R, C]     (bf16 operands; W as it lies, no transposed copy)
//
// The NN form of the forward kernel: W is staged like the weight gradient's X (reduction slow) and read transposed. Tiles that
// would leave CUs idle in a last round (or all of them, for few rows) are split over the reduction until the chip is full; the
// parts are written as fp32 and summed here (they stay in the L2 and the memory-side cache).
// =====================================================================================
// C of the tiles from `whole` on = sum of the parts, in order. Block: 8 rows of a tile, of 256 threads; 2 of 64 for a single row of
// tiles: few rows' parts through a few CUs' load paths take longer than their products (16 rows, 19 parts of 2560 columns: 3 us).
__global__ __launch_bounds__(256) void tgemm_sum_kernel(const TGArgs a) {
  const int lg = 31 - __clz(blockDim.x) - 5;  // rows of the block: 8 or 2
  const int rest = a.tiles_m * a.tiles_n - a.whole, t = blockIdx.x >> (8 - lg), wg = a.whole + t;
  const int band = wg / (TG_GROUP_M * a.tiles_n), first = band * TG_GROUP_M, rows = min(a.tiles_m - first, TG_GROUP_M);
  const int in_band = wg - band * TG_GROUP_M * a.tiles_n;
  const int row = ((blockIdx.x & ((256 >> lg) - 1)) << lg) + (threadIdx.x >> 5), col = (threadIdx.x & 31) * 8;
  const int m = (first + in_band % rows) * 256 + row, n = in_band / rows * 256 + col;
  if (m >= a.M || n >= a.N) return;
  const float* p = a.part + ((size_t)t << 16) + row * 256 + col;
  f32x4 v0 = *reinterpret_cast<const f32x4*>(p), v1 = *reinterpret_cast<const f32x4*>(p + 4);
  for (int s = 1; s < a.splits; s += 8) {  // eight parts requested at a time, the last few too
    f32x4 q0[8], q1[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (s + j < a.splits) {
        const float* q = p + ((size_t)(s + j) * rest << 16);
        q0[j] = *reinterpret_cast<const f32x4*>(q);
        q1[j] = *reinterpret_cast<const f32x4*>(q + 4);
      }
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (s + j < a.splits) {
        v0 += q0[j];
        v1 += q1[j];
      }
  }
  bf16_t* op = a.C + (size_t)m * a.ldc + n;
  *reinterpret_cast<bf16x4*>(op) = bf16x4{f2bf(v0[0]), f2bf(v0[1]), f2bf(v0[2]), f2bf(v0[3])};
  if (n + 8 <= a.N) *reinterpret_cast<bf16x4*>(op + 4) = bf16x4{f2bf(v1[0]), f2bf(v1[1]), f2bf(v1[2]), f2bf(v1[3])};
}

// The label's logit of every row, of the same products in the same order as the tiles above (and so with their bits): a wave's
// 16 rows against their 16 label rows of B, the diagonal of the result. out[m] = bf16 logit * inv_temp, 0 for a label outside
// [first, first + N).
__global__ __launch_bounds__(256) void tgemm_label_kernel(const bf16_t* __restrict__ A, long lda, const bf16_t* __restrict__ B,
                                                          long ldb, const int64_t* __restrict__ labels, int64_t first, int M,
                                                          int N, int K, float inv_temp, float* __restrict__ out) {
  const int lane = threadIdx.x & 63, fr = lane & 15, fq = lane >> 4;
  const int m0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 16;
  if (m0 >= M) return;
  const int m = min(m0 + fr, M - 1);
  const int64_t lab = labels[m] - first;
  const bool has = lab >= 0 && lab < N;
  const bf16_t* pa = A + (size_t)m * lda + fq * 8;
  const bf16_t* pb = B + (size_t)(has ? lab : 0) * ldb + fq * 8;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int k = 0; k < K; k += 32) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ld8(pb + k), ld8(pa + k), acc, 0, 0, 0);
  // lane (fr, fq) holds rows 4 fq .. 4 fq + 3 (labels) of column fr (token)
  const float v = (fr & 3) == 0 ? acc[0] : (fr & 3) == 1 ? acc[1] : (fr & 3) == 2 ? acc[2] : acc[3];
  if (fq == fr >> 2 && m0 + fr < M) out[m0 + fr] = has ? bf2f(f2bf(v)) * inv_temp : 0.f;
}

// part [3][cbs][M] of the statistics form -> largest logit, sum of exponentials and weighted sum of a row, of logits divided by
// the temperature. 32 rows a workgroup, the column blocks dealt to 32 threads each.
__global__ __launch_bounds__(1024) void tgemm_stats_kernel(const float* __restrict__ part, int cbs, int M, float scale,
                                                           float inv_temp, float* __restrict__ out_m, float* __restrict__ out_s,
                                                           float* __restrict__ out_w) {
#pragma clang fp contract(off)  // largest * scale is the rounded product that the tiles' sums are relative to
  __shared__ float red[3][32][33];
  const int r = threadIdx.x & 31, g = threadIdx.x >> 5, m = blockIdx.x * 32 + r;
  const size_t plane = (size_t)cbs * M;
  float mx = -INFINITY, s = 0.f, w = 0.f;
  auto merge = [&](float m2, float s2, float w2) {  // sums relative to 2^round(largest * scale); a side without anything adds nothing
    const float top = fmaxf(mx, m2), ref = top * scale;
    const float f1 = s == 0.f ? 0.f : __builtin_amdgcn_exp2f(mx * scale - ref);
    const float f2 = s2 == 0.f ? 0.f : __builtin_amdgcn_exp2f(m2 * scale - ref);
    s = s * f1 + s2 * f2;
    w = w * f1 + w2 * f2;
    mx = top;
  };
  if (m < M) {
#pragma unroll 4
    for (int cb = g; cb < cbs; cb += 32) {
      const float* p = part + (size_t)cb * M + m;
      merge(p[0], p[plane], p[2 * plane]);
    }
  }
  red[0][g][r] = mx;
  red[1][g][r] = s;
  red[2][g][r] = w;
  __syncthreads();
  if (g == 0 && m < M) {
    for (int i = 1; i < 32; ++i) merge(red[0][i][r], red[1][i][r], red[2][i][r]);
    const float ref = mx * scale, to = 1.f - 0.69314718f * fmaf(mx, scale, -ref);  // 2^(ref - largest * scale)
    out_m[m] = mx * inv_temp;
    out_s[m] = s * to;
    out_w[m] = w * to * inv_temp;
  }
}

}  // namespace

static void tgemm_sum_launch(const TGArgs& a, long tiles, hipStream_t st) {
  const int threads = a.tiles_m == 1 ? 64 : 256;
  hipLaunchKernelGGL(tgemm_sum_kernel, dim3((unsigned)(tiles * (8192 / threads))), dim3(threads), 0, st, a);
}

// C[M, N] = A[M, K] . B[N, K]^T (+ bias). Leading dimensions in elements (multiples of 8: 16-byte rows), K a multiple
// of 128, N a multiple of 4. Returns -1 for shapes outside that (the caller keeps its library path).
// One launch = min(tiles, max_blocks) persistent workgroups (256 = one per CU). splits > 1 (no bias): the tiles from `whole` on
// in parts, as for areal_tgemm_nn.
// gated = 1: B holds 2 N rows (gate rows, then up rows), C[M, N] = silu(A.gate^T) * (A.up^T), no bias.
static int tgemm_tn_launch(const void* A, long lda, const void* B, long ldb, void* C, long ldc, const void* bias, int M,
                           int N, int K, int max_blocks, int gated, float* part, int whole, int splits, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  if (K % 128 != 0 || K < 128 || N % 4 != 0 || lda % 8 != 0 || ldb % 8 != 0 || ldc % 4 != 0) return -1;
  if (((uintptr_t)A | (uintptr_t)B) % 16 != 0 || (uintptr_t)C % 8 != 0 || (bias && (uintptr_t)bias % 8 != 0)) return -1;
  if (gated && bias) return -1;
  const long tiles = (long)((M + 255) / 256) * (gated ? (N + 127) / 128 : (N + 255) / 256);
  const int pairs = K / 128;
  int chunk = pairs;
  if (splits == 1) {
    whole = (int)tiles;
  } else {  // (see areal_tgemm_nn)
    if (gated || bias || splits < 1 || splits > pairs || whole < 0 || whole >= tiles || whole % 256 != 0 || !part ||
        (uintptr_t)part % 16 != 0)
      return -1;
    chunk = (pairs + splits - 1) / splits;
    if ((pairs + chunk - 1) / chunk != splits) return -1;
  }
  const long items = whole + (tiles - whole) * splits;
  if (items > 0x7fffffffl - 256) return -1;
  TGArgs a{(const bf16_t*)A, lda, (const bf16_t*)B, ldb, (bf16_t*)C, ldc, (const bf16_t*)bias, M, N, K,
           (M + 255) / 256, gated ? (N + 127) / 128 : (N + 255) / 256, part, whole, splits, chunk, nullptr, 0};
  static bool attr_set = false;  // 160 KiB of dynamic LDS, 128 the gated form: above the default limit
  if (!attr_set) {
    HIP_RET(hipFuncSetAttribute((const void*)tgemm_kernel<0, false, false>, hipFuncAttributeMaxDynamicSharedMemorySize, TG_LDS + TG_OUT));
    HIP_RET(hipFuncSetAttribute((const void*)tgemm_kernel<1, false, false>, hipFuncAttributeMaxDynamicSharedMemorySize, TG_LDS));
    attr_set = true;
  }
  // max_blocks workgroups (a multiple of 8: block id mod 8 is the XCD for every tile of a block's sequence) walk the
  // tiles; 0 = one workgroup per tile
  if (max_blocks > 0 && max_blocks % 8 != 0) return -1;
  const dim3 grid((unsigned)(max_blocks > 0 ? std::min(items, (long)max_blocks) : items)), block(512);
  if (gated)
    hipLaunchKernelGGL((tgemm_kernel<1, false, false>), grid, block, TG_LDS, st, a);
  else
    hipLaunchKernelGGL((tgemm_kernel<0, false, false>), grid, block, TG_LDS + TG_OUT, st, a);
  if (splits > 1) tgemm_sum_launch(a, tiles - whole, st);
  return (int)hipGetLastError();
}

extern "C" int areal_tgemm_tn(const void* A, long lda, const void* B, long ldb, void* C, long ldc, const void* bias,
                              int M, int N, int K, int max_blocks, float* part, int whole, int splits, hipStream_t st) {
  return tgemm_tn_launch(A, lda, B, ldb, C, ldc, bias, M, N, K, max_blocks, 0, part, whole, splits, st);
}

// Statistics of the rows of logits A[M, K] . B[N, K]^T / temperature (rounded to bf16 before the division), which are not
// written: out_m the largest, out_s sum exp(z - largest), out_w the same weighted with z, out_tgt the label's (0 for labels
// outside [first, first + N)). part: 3 * ceil(N / 64) * M floats; inv_temp > 0. Returns -1 for shapes that areal_tgemm_tn
// does not take.
extern "C" int areal_tgemm_stats(const void* A, long lda, const void* B, long ldb, const int64_t* labels, long first, int M, int N,
                                 int K, float inv_temp, float* part, float* out_m, float* out_s, float* out_w, float* out_tgt,
                                 hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  if (K % 128 != 0 || K < 128 || N % 4 != 0 || lda % 8 != 0 || ldb % 8 != 0 || !(inv_temp > 0.f)) return -1;
  if (((uintptr_t)A | (uintptr_t)B) % 16 != 0 || !part) return -1;
  const long tiles = (long)((M + 255) / 256) * ((N + 255) / 256);
  if (tiles > 0x7fffffffl - 256) return -1;
  TGArgs a{(const bf16_t*)A, lda, (const bf16_t*)B, ldb, nullptr, 0, nullptr, M, N, K, (M + 255) / 256, (N + 255) / 256, part,
           (int)tiles, 1, K / 128, nullptr, 0, inv_temp * 1.4426950408889634f};
  static bool attr_set = false;  // 128 KiB of dynamic LDS: above the default limit
  if (!attr_set) {
    HIP_RET(hipFuncSetAttribute((const void*)tgemm_kernel<2, false, false>, hipFuncAttributeMaxDynamicSharedMemorySize, TG_LDS));
    attr_set = true;
  }
  hipLaunchKernelGGL((tgemm_kernel<2, false, false>), dim3((unsigned)std::min(tiles, 256l)), dim3(512), TG_LDS, st, a);
  hipLaunchKernelGGL(tgemm_label_kernel, dim3((unsigned)((M + 63) / 64)), dim3(256), 0, st, (const bf16_t*)A, lda, (const bf16_t*)B,
                     ldb, labels, (int64_t)first, M, N, K, inv_temp, out_tgt);
  hipLaunchKernelGGL(tgemm_stats_kernel, dim3((unsigned)((M + 31) / 32)), dim3(1024), 0, st, part, (N + 63) / 64, M, a.scale, inv_temp,
                     out_m, out_s, out_w);
  return (int)hipGetLastError();
}

// C[M, F] = silu(A . Wg^T) * (A . Wu^T) with W = [Wg; Wu] of shape [2 F, K] (the gate|up projection of a gated MLP and
// its activation in one kernel: the [M, 2 F] intermediate is never written). For forward passes that keep no
// activations (scoring, prefill).
extern "C" int areal_tgemm_swiglu(const void* A, long lda, const void* W, long ldw, void* C, long ldc, int M, int F,
                                  int K, int max_blocks, hipStream_t st) {
  return tgemm_tn_launch(A, lda, W, ldw, C, ldc, nullptr, M, F, K, max_blocks, 1, nullptr, 0, 1, st);
}

// dW[N, K] (fp32, leading dimension ldw) += dY[M, N]^T . X[M, K]. N a multiple of 128, K of 256, rows 16-byte aligned.
// The first `whole` tiles of 256 x 256 (a multiple of 256, or all of them: splits = 1) are reduced by one workgroup each, the
// others in `splits` parts; part: splits x 65536 floats for each of those. Every part has to have work, as for areal_tgemm_nn.
// A ragged last 128-token pair is filled up with zeros: handing its few tokens to a library GEMM
// instead reads and writes the whole fp32 gradient a second time (60 tokens: 51 us for 17920 x 1536, 507 us for the
// 151936 x 1536 LM head, 1.4 of the 9.2 ms of a pass over 700 tokens and 7 layers).
extern "C" int areal_tgemm_wgrad(const void* dY, long ldy, const void* X, long ldx, float* dW, long ldw, int M, int N,
                                 int K, int splits, int whole, float* part, hipStream_t st) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  if (N % 128 != 0 || K % 256 != 0 || ldy % 8 != 0 || ldx % 8 != 0) return -1;
  if (ldy < N || ldx < K) return -1;  // the loads end at the last row's last byte: rows must not overlap
  if (ldy > (1l << 24) || ldx > (1l << 24)) return -1;  // byte offsets of 64 rows: 32 bits
  if (((uintptr_t)dY | (uintptr_t)X) % 16 != 0 || (uintptr_t)dW % 4 != 0 || (uintptr_t)part % 16 != 0) return -1;
  const int pairs = (M - 1) / 128 + 1;
  const long tiles = (long)((N + 255) / 256) * (K / 256);
  if (splits < 1 || splits > pairs || whole < 0 || whole > tiles) return -1;
  if (splits == 1 ? whole != tiles : whole % 256 != 0 || whole == tiles || !part) return -1;
  const int chunk = (pairs + splits - 1) / splits;
  if ((pairs + chunk - 1) / chunk != splits) return -1;
  const long nblocks = whole + (tiles - whole) * splits;
  if (nblocks > 0x7fffffffl || (tiles - whole) > (0x7fffffffl >> 5)) return -1;
  TWArgs a{(const bf16_t*)dY, ldy, (const bf16_t*)X, ldx, dW, ldw, M, N, K, (N + 255) / 256, K / 256, pairs, whole, splits, chunk, part, nullptr, 0};
  static bool attr_set = false;
  if (!attr_set) {
    HIP_RET(hipFuncSetAttribute((const void*)tgemm_wgrad_kernel<false, false>, hipFuncAttributeMaxDynamicSharedMemorySize, TG_LDS));
    HIP_RET(hipFuncSetAttribute((const void*)tgemm_wgrad_kernel<false, true>, hipFuncAttributeMaxDynamicSharedMemorySize, TG_LDS));
    attr_set = true;
  }
  if ((long)N * K >= TG_STREAM)
    hipLaunchKernelGGL((tgemm_wgrad_kernel<false, true>), dim3((unsigned)nblocks), dim3(512), TG_LDS, st, a);
  else
    hipLaunchKernelGGL((tgemm_wgrad_kernel<false, false>), dim3((unsigned)nblocks), dim3(512), TG_LDS, st, a);
  if (splits > 1) hipLaunchKernelGGL(tgemm_wgrad_sum_kernel, dim3((unsigned)(tiles - whole) * 32), dim3(256), 0, st, a);
  return (int)hipGetLastError();
}

// The same for few tokens (tiles of 128 x 128, no parts); K a multiple of 128.
extern "C" int areal_tgemm_wgrad_few(const void* dY, long ldy, const void* X, long ldx, float* dW, long ldw, int M, int N, int K,
                                     hipStream_t st) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  if (N % 128 != 0 || K % 128 != 0 || ldy % 8 != 0 || ldx % 8 != 0) return -1;
  if (ldy < N || ldx < K || ldy > (1l << 24) || ldx > (1l << 24)) return -1;  // (as above)
  if (((uintptr_t)dY | (uintptr_t)X) % 16 != 0 || (uintptr_t)dW % 4 != 0) return -1;
  const long tiles = (long)(N / 128) * (K / 128);
  if (tiles > 0x7fffffffl) return -1;
  const TWArgs a{(const bf16_t*)dY, ldy, (const bf16_t*)X, ldx, dW, ldw, M, N, K, N / 128, K / 128, 0, 0, 1, 0, nullptr, nullptr, 0};
  if (tiles <= 768)  // three a CU
    hipLaunchKernelGGL((tgemm_wgrad_few_kernel<false, 3>), dim3((unsigned)tiles), dim3(256), 3 * TWF_STAGE, st, a);
  else
    hipLaunchKernelGGL((tgemm_wgrad_few_kernel<false, 2>), dim3((unsigned)tiles), dim3(256), 2 * TWF_STAGE, st, a);
  return (int)hipGetLastError();
}

// dX[M, C] = dY[M, R] . W[R, C]; R a multiple of 128, C of 256, rows 16-byte aligned. The first `whole` tiles of 256 x 256 (a
// multiple of 256, so that the parts start a round, or all of them: splits = 1) are reduced by one workgroup, the others in
// `splits` parts. part: splits x 65536 floats for each of those. Every part has to have work: with P = R / 128,
// ceil(P / ceil(P / splits)) == splits (12 pairs in 5 parts are 4).
extern "C" int areal_tgemm_nn(const void* dY, long ldy, const void* W, long ldw, void* dX, long ldx, float* part, int whole,
                              int splits, int M, int R, int C, hipStream_t st) {
  if (M <= 0 || R <= 0 || C <= 0) return R <= 0 && M > 0 && C > 0 ? -1 : 0;
  if (R % 128 != 0 || C % 256 != 0 || ldy % 8 != 0 || ldw % 8 != 0 || ldx % 4 != 0) return -1;
  if (((uintptr_t)dY | (uintptr_t)W) % 16 != 0 || (uintptr_t)dX % 8 != 0 || (uintptr_t)part % 16 != 0) return -1;
  if (ldy < R || ldw < C || ldx < C || ldy > (1l << 22) || ldw > (1l << 24)) return -1;
  const int tiles_m = (M + 255) / 256, pairs = R / 128;
  const long tiles = (long)tiles_m * (C / 256);
  if (tiles > 0x7fffffffl || splits < 1 || splits > pairs || whole < 0 || whole > tiles) return -1;
  if (splits == 1 ? whole != tiles : whole % 256 != 0 || whole == tiles || !part) return -1;
  const int chunk = (pairs + splits - 1) / splits;
  if ((pairs + chunk - 1) / chunk != splits) return -1;  // a part without work would leave its sums unwritten
  const long items = whole + (tiles - whole) * splits;
  if (items > 0x7fffffffl - 256) return -1;
  TGArgs a{(const bf16_t*)dY, ldy, (const bf16_t*)W, ldw, (bf16_t*)dX, ldx, nullptr, M, C, R, tiles_m, C / 256,
           part, whole, splits, chunk, nullptr, 0};
  static bool attr_set = false;
  if (!attr_set) {
    HIP_RET(hipFuncSetAttribute((const void*)tgemm_kernel<0, true, false>, hipFuncAttributeMaxDynamicSharedMemorySize, TG_LDS + TG_OUT));
    attr_set = true;
  }
  hipLaunchKernelGGL((tgemm_kernel<0, true, false>), dim3((unsigned)std::min(items, 256l)), dim3(512), TG_LDS + TG_OUT, st, a);
  if (splits > 1) tgemm_sum_launch(a, tiles - whole, st);
  return (int)hipGetLastError();
}

// ---- routed experts: rows sorted by expert, offsets [E + 1] on the device. table: 4 (T / 256 + E + 1) ints of scratch.
// nn = 0: C[t, N] = A[t, K] . B[e, N, K]^T, K a multiple of 128, N of 8; nn = 1: C[t, N] = A[t, K] . B[e, K, N], N of 256.
extern "C" int areal_tgemm_grouped(const void* A, const void* B, void* C, const int* offsets, int* table, int T, int E, int N,
                                   int K, long stride, int nn, hipStream_t st) {
  if (T <= 0 || E <= 0) return 0;
  if (K % 128 != 0 || K < 128 || N <= 0 || N % (nn ? 256 : 8) != 0 || stride % 8 != 0) return -1;
  if (((uintptr_t)A | (uintptr_t)B | (uintptr_t)C | (uintptr_t)table) % 16 != 0) return -1;
  const int tiles_n = (N + 255) / 256;
  const long most = ((long)T / 256 + E) * tiles_n;  // (an expert's last tile may be partly empty)
  if (most > 0x7fffffffl - 256) return -1;
  hipLaunchKernelGGL(tgemm_table_kernel, dim3(1), dim3(256), 0, st, offsets, E, (int4*)table);
  TGArgs a{(const bf16_t*)A, K, (const bf16_t*)B, nn ? N : K, (bf16_t*)C, N, nullptr, T, N, K, 0, tiles_n,
           nullptr, 0, 1, 0, (const int4*)table, stride};
  static bool attr_set = false;
  if (!attr_set) {
    HIP_RET(hipFuncSetAttribute((const void*)tgemm_kernel<0, false, true>, hipFuncAttributeMaxDynamicSharedMemorySize, TG_LDS + TG_OUT));
    HIP_RET(hipFuncSetAttribute((const void*)tgemm_kernel<0, true, true>, hipFuncAttributeMaxDynamicSharedMemorySize, TG_LDS + TG_OUT));
    attr_set = true;
  }
  const dim3 grid((unsigned)std::min(most, 256l)), block(512);
  if (nn)
    hipLaunchKernelGGL((tgemm_kernel<0, true, true>), grid, block, TG_LDS + TG_OUT, st, a);
  else
    hipLaunchKernelGGL((tgemm_kernel<0, false, true>), grid, block, TG_LDS + TG_OUT, st, a);
  return (int)hipGetLastError();
}

// dW[e, N, K] (fp32, experts `stride` elements apart) += dY[t, N]^T . X[t, K] over each expert's rows; N a multiple of 128, K
// of 256.
extern "C" int areal_tgemm_grouped_wgrad(const void* dY, const void* X, float* dW, const int* offsets, int E, int N, int K,
                                         long stride, hipStream_t st) {
  if (E <= 0) return 0;
  if (N <= 0 || K <= 0 || N % 128 != 0 || K % 256 != 0 || N > (1 << 24) || K > (1 << 24)) return -1;
  if (((uintptr_t)dY | (uintptr_t)X) % 16 != 0 || (uintptr_t)dW % 4 != 0) return -1;
  const int tiles_n = (N + 255) / 256, tiles_k = K / 256;
  const long blocks = (long)tiles_n * tiles_k * E;
  if (blocks > 0x7fffffffl) return -1;
  TWArgs a{(const bf16_t*)dY, N, (const bf16_t*)X, K, dW, K, 0, N, K, tiles_n, tiles_k, 0, (int)blocks, 1, 0, nullptr, offsets, stride};
  static bool attr_set = false;
  if (!attr_set) {
    HIP_RET(hipFuncSetAttribute((const void*)tgemm_wgrad_kernel<true, false>, hipFuncAttributeMaxDynamicSharedMemorySize, TG_LDS));
    HIP_RET(hipFuncSetAttribute((const void*)tgemm_wgrad_kernel<true, true>, hipFuncAttributeMaxDynamicSharedMemorySize, TG_LDS));
    attr_set = true;
  }
  if ((long)E * N * K >= TG_STREAM)
    hipLaunchKernelGGL((tgemm_wgrad_kernel<true, true>), dim3((unsigned)blocks), dim3(512), TG_LDS, st, a);
  else
    hipLaunchKernelGGL((tgemm_wgrad_kernel<true, false>), dim3((unsigned)blocks), dim3(512), TG_LDS, st, a);
  return (int)hipGetLastError();
}

// The same for few rows an expert (tiles of 128 x 128), `most` at most; K a multiple of 128. `spread`: each expert's tiles are dealt to all XCDs.
extern "C" int areal_tgemm_grouped_wgrad_few(const void* dY, const void* X, float* dW, const int* offsets, int most, int E, int N, int K,
                                             long stride, int spread, hipStream_t st) {
  if (E <= 0) return 0;
  if (N <= 0 || K <= 0 || N % 128 != 0 || K % 128 != 0 || N > (1 << 24) || K > (1 << 24)) return -1;
  if (((uintptr_t)dY | (uintptr_t)X) % 16 != 0 || (uintptr_t)dW % 4 != 0) return -1;
  const long per = (long)(N / 128) * (K / 128), tiles = per * E;
  if (tiles > 0x7fffffffl) return -1;
  // Few rows' operands fit the L2 in any order, and tile after tile along the gradient's rows the memory is read and written in
  // longer pieces: us in bands of 1 / 8 tile rows, 8 experts of 4096 x 14336, 16 / 64 / 128 / 200 / 400 rows 695 / 723, 696 / 727, 696 / 724, 730
  // / 725, 911 / 747; 128 of 1536 x 2048 525 / 559, 521 / 546, 517 / 540, 523 / 552, 641 / 687; 16 of 2048 x 7168 343 / 361, 341 / 361,
  // 342 / 360, 344 / 360, 449 / 377; all of 254 / 508 / 1016 rows with one of the first 193 / 194, 221 / 203, 786 / 760.
  const int band = most <= 256 ? 1 : 8;
  const TWArgs a{(const bf16_t*)dY, N, (const bf16_t*)X, K, dW, K, 0, N, K, N / 128, K / 128, 0, 0, 1, spread, nullptr, offsets, stride, band};
  hipLaunchKernelGGL((tgemm_wgrad_few_kernel<true, 2>), dim3((unsigned)tiles), dim3(256), 2 * TWF_STAGE, st, a);
  return (int)hipGetLastError();
}
