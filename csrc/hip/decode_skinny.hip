// The projections of a decoder layer for a decode step of at most 8 rows, on gfx950: Y[M, N] = X[M, K] W[N, K]^T with
// what surrounds it in the same launch, five launches a layer instead of eight:
//
//   qkv      RMSNorm of the residual stream, the projection, bias, rotation, KV-cache write
//   (paged attention)
//   o        the projection + residual sum
//   gate|up  RMSNorm, the projection, gated activation
//   down     the projection + residual sum
//
// What bounds it: streaming the weights (55 MB from 256 workgroups that only load: 9.9 us; 6 TB/s in steady state), and as
// much the chain of dependent launches: a row kernel that sums split-K slabs and normalises takes 4.4 us for a few KB. So
// a workgroup owns its columns over ALL of K - no slabs, nothing to hand over - and normalises the rows itself, under the
// latency of its weight loads. One workgroup a CU: N / 256 columns each (o, down of Qwen2-1.5B: 6, gate|up: 35 + 35, qkv:
// 4 rotated pairs).
//
//   * one and two rows: no matrix cores. A packed dot product (v_dot2_f32_bf16: two products added to an fp32 sum) per
//     pair of weights and row keeps up with memory, and a wave reads 1 KiB of ONE weight row per load instruction; as
//     matrix operands (16 rows x 64 bytes a load) the same bytes take 10.8 instead of 9.2 us to load;
//   * three to eight rows: matrix cores (with three rows the dot products take as long as the loads, with eight twice as
//     long: 2.3 ms a step), but the long rows of a narrow down projection (areal_skinny_residual); from nine rows on the split-K path is
//     as fast;
//   * 8 waves: WK along K, 8 / WK along the rows, WK so that a wave's share of K is at most 3 x 64 pieces of 16 bytes
//     (K = 1536: WK = 1, K = 8960: WK = 8); the wave's share of the activations stays in registers for all its rows;
//   * two sets of RB weight rows in registers: all loads of gate|up, o and down of Qwen2-1.5B are in flight at once;
//   * lane sums are folded two values at a time by permlane swaps; the waves' sums meet in LDS and are added in the order
//     of the waves: results do not depend on timing.
//
// Rounding points are those of the split-K path (csrc/hip/decode_gemm.hip): normalised rows, projection and residual
// sum in bf16, sums in fp32.
//
// Measured (Qwen2-1.5B, 640-token contexts, captured decode step of 28 layers), split-K path / this: 1 row 1.24 / 1.07 ms, 2 rows 1.26 /
// 1.19, 3 rows 1.27 / 1.26, 4 rows 1.28 / 1.27, 6 rows 1.29 / 1.38 (which rows take it: ModelRunner). One row: gate|up 11.8 us, down 7.3, o 3.2,
// qkv 4.4.
#include "common.hpp"

namespace {

enum { SK_RES = 0, SK_GATED = 1, SK_QKV = 2 };
constexpr int WAVES = 8, THREADS = 64 * WAVES;

struct SKArgs {
  const bf16_t* X;   // [M, K] rows of stride xs: activations, or the residual stream (NORM)
  const bf16_t* W;   // [N, K]
  const bf16_t* nw;  // norm weight [K]
  const bf16_t* res; // SK_RES: residual rows [M, N] (contiguous) or null
  bf16_t* Y;         // SK_RES: [M, N]; SK_GATED: [M, N / 2]; SK_QKV: rotated q [M, Hq, D]
  int64_t xs;
  int M, N, K, cols; // cols: columns of a workgroup (SK_GATED: of either half; SK_QKV: rotated pairs)
  float eps;
  int gemma, act;
  const bf16_t* bias;
  const int* pos;
  const int64_t* slots;
  const float* cos_t;
  const float* sin_t;
  void* kcache;
  void* vcache;
  int Hq, Hkv, D, max_pos, do_rope, fp8;
  // PARTS: what the decode attention has left of X: partial results rows[0].x .. + rows[0].y, or X itself where that is one
  const float *part_o, *part_ml;
  const int2* rows;
  int d_shift;       // log2 of the head size
  unsigned per_inv;  // qkv_rows: reciprocal of the column blocks of a head
};

DEVINL float sk_gate(float x, int act) {
  if (act == 0) return x / (1.f + __expf(-x));
  const float inner = 0.7978845608028654f * (x + 0.044715f * x * x * x);
  const float e = __expf(-2.f * fabsf(inner));
  return 0.5f * x * (1.f + copysignf((1.f - e) / (1.f + e), inner));
}

constexpr int P = 3;  // passes of 64 16-byte pieces that a wave makes over its share of K

// Sum over the 64 lanes of each of V values; value v ends up in the lanes of row (v % 4 -> 0, 2, 1, 3) of out[v / 4].
template <int V>
DEVINL void lane_sums(const float (&x)[V], float (&out)[(V + 3) / 4]) {
#pragma unroll
  for (int j = 0; j < (V + 3) / 4; ++j) {
    float y[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const unsigned a = __float_as_uint(4 * j + 2 * h < V ? x[4 * j + 2 * h < V ? 4 * j + 2 * h : 0] : 0.f);
      const unsigned b = __float_as_uint(4 * j + 2 * h + 1 < V ? x[4 * j + 2 * h + 1 < V ? 4 * j + 2 * h + 1 : 0] : 0.f);
      const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);  // {a low, b low}, {a high, b high}
      y[h] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(y[0]), __float_as_uint(y[1]), false, false);
    float z = __uint_as_float(r[0]) + __uint_as_float(r[1]);
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) z += __shfl_xor(z, o, 64);
    out[j] = z;
  }
}

DEVINL float dot8(bf16x8 a, bf16x8 b, float c) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    c = __builtin_amdgcn_fdot2_f32_bf16((bf16x2){a[2 * i], a[2 * i + 1]}, (bf16x2){b[2 * i], b[2 * i + 1]}, c, false);
  return c;
}

// Members d and d + D / 2 of a head of row m: bias (0: none), rotation (c = 1, s = 0 where none is wanted; V heads have none), q to
// a.Y, k and v to their page.
DEVINL void put_pair(const SKArgs& a, int head, int d, int m, float lo, float hi, float bias_lo, float bias_hi, float c, float s,
                     int64_t slot) {
  const int half = a.D >> 1;
  lo = bf2f(f2bf(lo + bias_lo));  // the unfused path carries the projection as a bf16 tensor
  hi = bf2f(f2bf(hi + bias_hi));
  if (a.do_rope && head < a.Hq + a.Hkv) {
    const float x = lo;  // (which product is rounded by itself is written out: left to the compiler it changes with the code around it)
    lo = fmaf(x, c, -(hi * s));
    hi = fmaf(hi, c, x * s);
  }
  if (head < a.Hq) {
    bf16_t* q = a.Y + ((size_t)m * a.Hq + head) * a.D + d;
    q[0] = f2bf(lo);
    q[half] = f2bf(hi);
    return;
  }
  if (slot < 0) return;
  const int64_t page = slot / 32;
  const int off = (int)(slot % 32);
  if (head < a.Hq + a.Hkv) {
    const size_t at = (((size_t)page * a.Hkv + head - a.Hq) * 32 + off) * a.D + d;
    st1_cache(a.kcache, at, bf2f(f2bf(lo)), a.fp8);  // fp8: from the bf16 value, as the other writers
    st1_cache(a.kcache, at + half, bf2f(f2bf(hi)), a.fp8);
  } else {
    const size_t at = (((size_t)page * a.Hkv + head - a.Hq - a.Hkv) * a.D + d) * 32 + off;
    st1_cache(a.vcache, at, lo, a.fp8);
    st1_cache(a.vcache, at + (size_t)half * 32, hi, a.fp8);
  }
}

// What follows the projection; sum(j, h, m): the fp32 sum of column j (SK_GATED: of half h; SK_QKV: member h of pair j) of
// row m, read from LDS. SK_RES: one result a thread, of column rj and row rm, and its residual.
template <int MODE, typename Sum>
DEVINL void finish(const SKArgs& a, int rj, int rm, float res, Sum sum) {
  if (MODE == SK_RES) {
    const int n = blockIdx.x * a.cols + rj;
    if (rm >= a.M || n >= a.N) return;
    float s = sum(rj, 0, rm);
    if (a.res) s = bf2f(f2bf(s)) + res;
    a.Y[(size_t)rm * a.N + n] = f2bf(s);
  } else if (MODE == SK_GATED) {
    const int F = a.N >> 1;
    for (int i = threadIdx.x; i < a.cols * a.M; i += THREADS) {
      const int j = i % a.cols, m = i / a.cols, n = blockIdx.x * a.cols + j;
      if (n >= F) continue;
      // gate / up rounded to bf16 first: the values an unfused bf16 GEMM output would carry
      const float g = bf2f(f2bf(sum(j, 0, m))), u = bf2f(f2bf(sum(j, 1, m)));
      a.Y[(size_t)m * F + n] = f2bf(sk_gate(g, a.act) * u);
    }
  } else {
    const int half = a.D >> 1, per = half / a.cols;
    const int head = blockIdx.x / per, d0 = (blockIdx.x % per) * a.cols;
    for (int i = threadIdx.x; i < a.cols * a.M; i += THREADS) {
      const int j = i % a.cols, m = i / a.cols, d = d0 + j;
      float c = 1.f, s = 0.f;
      if (a.do_rope && head < a.Hq + a.Hkv) {
        int p = a.pos[m];
        p = p < 0 ? 0 : (p >= a.max_pos ? a.max_pos - 1 : p);
        c = a.cos_t[(size_t)p * half + d];
        s = a.sin_t[(size_t)p * half + d];
      }
      put_pair(a, head, d, m, sum(j, 0, m), sum(j, 1, m), a.bias ? bf2f(a.bias[head * a.D + d]) : 0.f,
               a.bias ? bf2f(a.bias[head * a.D + d + half]) : 0.f, c, s, head < a.Hq ? -1 : a.slots[m]);
    }
  }
}

// One and two rows, with SK_RES up to eight. MT: rows of X (a.M = MT); RB: weight rows of a register set; WK: waves along K; NORM: X is normalised first;
// TURNS: K > WK P 512, the waves go over their share more than once (not with NORM). Grid: workgroups (SK_QKV: of a head, heads).
// A launch is a few microseconds long, so what stands ahead of its first load counts: the waves' split is a template parameter and a
// wave's weight rows are one pointer and a step (rows of a pair, gate | up or the members of a rotation, belong to neighbouring
// rows j of the workgroup). With both worked out from arguments it was 270 (o) to 500 (gate|up) instructions, 30 to 60 now. What the
// results need besides the sums is asked for with the operands. Captured, cold weights, 1536 wide, us a launch before / now, one
// row: qkv 5.24 / 4.40, o 3.82 / 3.16, gate|up 12.86 / 11.81 (a bare stream of these 55 MB: 10.4), down 8.02 / 7.28; two rows: 5.74 /
// 5.24, 4.18 / 3.44, 13.8 / 12.9, 8.55 / 7.95. 8 steps of 28 layers at one row 9.50 -> 8.76 ms.
// PARTS (o): X is combined here from the partial results of the decode attention, in the order and with the roundings that it would
// combine them with itself: every workgroup reads all of them (30 KB at 640 tokens) ahead of its weights, where the attention's
// last workgroup of a row waits for its stores, a counter, the sums and the results, one trip past the L2 after the other. A row with a
// single partial result is read as the attention has written it. Captured, attention and o, 12 heads of 128 on 2, us apart / so: 100 / 300 /
// 640 / 1900 / 6000 / 20000 tokens 7.7 / 7.8, 10.2 / 8.5, 10.3 / 8.9, 12.1 / 10.9, 14.5 / 13.1, 20.5 / 18.8.
template <int MT, int RB, int WK, bool NORM, int MODE, bool TURNS, bool PARTS>
__global__ __launch_bounds__(THREADS) void skinny_dot_kernel(const SKArgs a) {
  constexpr int NWR = WAVES / WK;
  constexpr bool PAIRED = MODE != SK_RES;
  extern __shared__ __attribute__((aligned(16))) float rf[];  // [WK][rows of the workgroup][MT]
  __shared__ float sq[WAVES][MT];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wk = wave & (WK - 1), wr = wave / WK;
  const int nrows = PAIRED ? 2 * a.cols : a.cols;
  // row j of the workgroup: row b0 + j of W, PAIRED: b0 + j / 2 + (j % 2) second; `have` of them exist
  int b0, second = 0, have = nrows;
  if (MODE == SK_QKV) {
    second = a.D >> 1;
    b0 = blockIdx.y * a.D + blockIdx.x * a.cols;
  } else {
    const int F = MODE == SK_GATED ? a.N >> 1 : a.N;
    if (MODE == SK_GATED) second = F;
    b0 = blockIdx.x * a.cols;
    have = min(a.cols, F - b0) * (PAIRED ? 2 : 1);
  }
  const int pieces = a.K >> 3;                // 16-byte pieces of a row
  const int seg = (pieces + WK - 1) / WK;     // of a wave's share
  const size_t pitch = (size_t)a.K * sizeof(bf16_t);
  const char* row = reinterpret_cast<const char*>(a.W) + (size_t)(b0 + (PAIRED ? wr / 2 + (wr & 1) * second : wr)) * pitch;

  // this thread's result: column (SK_QKV: pair) j of row m
  int m = 0;
#pragma unroll
  for (int i = 1; i < MT; ++i) m += (int)threadIdx.x >= i * a.cols;
  const int j = threadIdx.x - m * a.cols;
  const int jc = min(j, (PAIRED ? have >> 1 : have) - 1);
  float res = 0.f, blo = 0.f, bhi = 0.f, c = 1.f, s = 0.f;
  int64_t slot = -1;

  // PARTS: four values a thread and turn, the first eight partial results of the first turn on their way ahead of the weights
  constexpr int PT = 4 * THREADS;
  f32x4 po[8];
  float2 pml[8];
  int first_part = 0, nparts = 0;
  auto fetch_parts = [&](int col, int k0) __attribute__((always_inline)) {
    const float* o = a.part_o + (size_t)(first_part + k0) * a.K + col;
    const float* ml = a.part_ml + ((size_t)(first_part + k0) * (a.K >> a.d_shift) + (col >> a.d_shift)) * 2;
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (k0 + k < nparts) {  // the same for all lanes
        po[k] = *reinterpret_cast<const f32x4*>(o + (size_t)k * a.K);
        pml[k] = *reinterpret_cast<const float2*>(ml + (size_t)k * (a.K >> a.d_shift) * 2);
      }
  };
  bf16_t* xs = reinterpret_cast<bf16_t*>(rf + (WK * nrows * MT + 3) / 4 * 4);  // [K]
  if constexpr (PARTS) {
    static_assert(MT == 1);
    const int2 r = a.rows[0];
    first_part = r.x;
    nparts = r.y;
    if (nparts > 1 && (int)threadIdx.x * 4 < a.K) fetch_parts(threadIdx.x * 4, 0);
    __builtin_amdgcn_sched_barrier(0);
  }

  for (int s0 = 0; s0 < (TURNS ? seg : 1); s0 += 64 * P) {
    unsigned at[P];  // this lane's pieces, in bytes
    bool ok[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int in = s0 + 64 * p + lane;
      ok[p] = in < seg && wk * seg + in < pieces;
      at[p] = (ok[p] ? wk * seg + in : 0) * 16;
    }
    bf16x8 xv[MT][P], nv[NORM ? P : 1];
    if (!PARTS || nparts <= 1)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int p = 0; p < P; ++p)
        xv[i][p] = *reinterpret_cast<const bf16x8*>(reinterpret_cast<const char*>(a.X + i * a.xs) + at[p]);
    if (NORM)
#pragma unroll
      for (int p = 0; p < P; ++p) nv[p] = *reinterpret_cast<const bf16x8*>(reinterpret_cast<const char*>(a.nw) + at[p]);
    __builtin_amdgcn_sched_barrier(0);  // ahead of the weights: loads return in order

    bf16x8 wv[2][RB][P];
    const char* next = row;
    auto load = [&](int set, int first) __attribute__((always_inline)) {  // the rows behind those of the last call
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        if (wr + NWR * (first + i) < have)  // the same for all lanes
#pragma unroll
          for (int p = 0; p < P; ++p) wv[set][i][p] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(next + at[p]));
        if (!PAIRED) next += NWR * pitch;
        else if (NWR > 1) next += NWR / 2 * pitch;
        else next += (set * RB + i) & 1 ? pitch - second * pitch : second * pitch;
      }
    };
    load(0, 0);
    load(1, RB);
    __builtin_amdgcn_sched_barrier(0);
    if (s0 == 0) {
      if (MODE == SK_RES && a.res) res = bf2f(a.res[(size_t)m * a.N + b0 + jc]);
      if (MODE == SK_QKV) {
        const int head = blockIdx.y, half = a.D >> 1, d = blockIdx.x * a.cols + jc;
        if (a.bias) {
          blo = bf2f(a.bias[head * a.D + d]);
          bhi = bf2f(a.bias[head * a.D + d + half]);
        }
        if (head >= a.Hq) slot = a.slots[m];
        if (a.do_rope && head < a.Hq + a.Hkv) {
          int p = a.pos[m];
          p = p < 0 ? 0 : (p >= a.max_pos ? a.max_pos - 1 : p);
          c = a.cos_t[(size_t)p * half + d];
          s = a.sin_t[(size_t)p * half + d];
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);

    if (PARTS && nparts > 1) {
      if (s0 == 0) {
        for (int col = threadIdx.x * 4; col < a.K; col += PT) {
          float mm = -INFINITY, ll = 0.f;
          f32x4 acc = {0.f, 0.f, 0.f, 0.f};
          for (int k0 = 0; k0 < nparts; k0 += 8) {
            if (k0 > 0 || col >= PT) fetch_parts(col, k0);
            float mn = mm;
#pragma unroll
            for (int k = 0; k < 8; ++k)
              if (k0 + k < nparts) mn = fmaxf(mn, pml[k].x);
            const float f0 = mm == -INFINITY ? 0.f : fast_exp2(mm - mn);
            if (k0 > 0) {
              acc *= f0;
              ll *= f0;
            }
            mm = mn;
#pragma unroll
            for (int k = 0; k < 8; ++k)
              if (k0 + k < nparts) {
                const float f = pml[k].x == -INFINITY ? 0.f : fast_exp2(pml[k].x - mn);
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] += po[k][e] * f;
                ll += pml[k].y * f;
              }
          }
          bf16x4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = f2bf(ll > 0.f ? acc[e] / ll : 0.f);
          *reinterpret_cast<bf16x4*>(xs + col) = o;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
#pragma unroll
      for (int p = 0; p < P; ++p) xv[0][p] = *reinterpret_cast<const bf16x8*>(reinterpret_cast<const char*>(xs) + at[p]);
    }

    // pieces beyond the wave's share count as zeros
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int i = 0; i < MT; ++i)
        if (!ok[p]) xv[i][p] = bf16x8{};
    if (NORM) {  // every wave normalises its share for itself; with one wave along K no other is asked
      float ss[MT], fold[(MT + 3) / 4];
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        ss[i] = 0.f;
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
          for (int e = 0; e < 8; ++e) ss[i] += bf2f(xv[i][p][e]) * bf2f(xv[i][p][e]);
      }
      lane_sums<MT>(ss, fold);
#pragma unroll
      for (int i = 0; i < MT; ++i) {  // value i sits in the lanes of row {0, 2, 1, 3}[i % 4]
        constexpr int row_of[4] = {0, 2, 1, 3};
        ss[i] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(fold[i >> 2]), 16 * row_of[i & 3]));
      }
      if (WK > 1) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
          if (lane == i) sq[wave][i] = ss[i];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          float t = 0.f;
          for (int w = 0; w < WK; ++w) t += sq[wave - wk + w][i];
          ss[i] = t;
        }
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const float rstd = rsqrtf(ss[i] / (float)a.K + a.eps);
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
          for (int e = 0; e < 8; ++e)
            xv[i][p][e] = f2bf(bf2f(xv[i][p][e]) * rstd * (bf2f(nv[p][e]) + (a.gemma ? 1.f : 0.f)));
      }
    }

    auto multiply = [&](int set, int first) __attribute__((always_inline)) {
      float acc[RB * MT], fold[(RB * MT + 3) / 4];
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int k = 0; k < MT; ++k) {
          acc[i * MT + k] = 0.f;
#pragma unroll
          for (int p = 0; p < P; ++p) acc[i * MT + k] = dot8(wv[set][i][p], xv[k][p], acc[i * MT + k]);
        }
      lane_sums<RB * MT>(acc, fold);
      if ((lane & 15) == 0) {
        const int g = lane >> 4, in4 = g == 1 ? 2 : g == 2 ? 1 : g;  // which of four values this row of lanes holds
#pragma unroll
        for (int f = 0; f < (RB * MT + 3) / 4; ++f) {
          const int v = 4 * f + in4, r = wr + NWR * (first + v / MT);
          if (v < RB * MT && r < nrows) {
            float* d = rf + ((size_t)wk * nrows + r) * MT + v % MT;
            *d = !TURNS || s0 == 0 ? fold[f] : *d + fold[f];
          }
        }
      }
    };
    for (int first = 0; wr + NWR * first < nrows; first += 2 * RB) {
#pragma unroll
      for (int set = 0; set < 2; ++set) {
        if (wr + NWR * (first + set * RB) < nrows) {
          multiply(set, first + set * RB);
          if (wr + NWR * (first + (set + 2) * RB) < nrows) load(set, first + (set + 2) * RB);
        }
      }
    }
  }
  __syncthreads();
  if ((int)threadIdx.x >= MT * a.cols || j != jc) return;
  auto sum = [&](int h) __attribute__((always_inline)) {
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < WK; ++w) t += rf[((size_t)w * nrows + (PAIRED ? 2 * j + h : j)) * MT + m];
    return t;
  };
  if (MODE == SK_RES) {
    float t = sum(0);
    if (a.res) t = bf2f(f2bf(t)) + res;
    a.Y[(size_t)m * a.N + b0 + j] = f2bf(t);
  } else if (MODE == SK_GATED) {
    // gate / up rounded to bf16 first: the values an unfused bf16 GEMM output would carry
    const float g = bf2f(f2bf(sum(0))), u = bf2f(f2bf(sum(1)));
    a.Y[(size_t)m * (a.N >> 1) + b0 + j] = f2bf(sk_gate(g, a.act) * u);
  } else {
    put_pair(a, blockIdx.y, blockIdx.x * a.cols + j, m, sum(0), sum(1), blo, bhi, c, s, slot);
  }
}

// Three to eight rows, on the matrix cores: CT 16-row weight tiles of a workgroup (SK_GATED: gate tiles, then as many up
// tiles), U: 64-deep chunks of K a wave has in flight (chunk c belongs to wave c mod 8), PRE: and as many more, in a second
// set of registers.
template <int CT, int U, bool PRE, bool NORM, int MODE>
__global__ __launch_bounds__(THREADS) void skinny_mfma_kernel(const SKArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  bf16_t* xn = reinterpret_cast<bf16_t*>(smem);  // normalised rows [M][K + 8]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, kq = lane >> 4;  // operand row (weights: column of Y; activations: row of Y), 8 k's each
  const int nchunk = a.K >> 6;
  const int mine = wave < nchunk ? (nchunk - wave + WAVES - 1) / WAVES : 0;

  // wave m normalises row m: its first pieces are loaded ahead of the weights, loads return in order
  bf16x8 hv[P], gv[P];
  if (NORM && wave < a.M) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int c = (lane + 64 * p) * 8;
      if (c < a.K) {
        hv[p] = ld8(a.X + (size_t)wave * a.xs + c);
        gv[p] = ld8(a.nw + c);
      }
    }
  }
  __builtin_amdgcn_sched_barrier(0);

  const bf16_t* wp[CT];  // this lane's weight rows; lanes without one repeat the workgroup's first: the same cache lines,
                         // and results that are not stored. Lanes without an activation row likewise
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    int row;
    if (MODE == SK_GATED) {
      const int j = 16 * (ct % (CT / 2)) + r, F = a.N >> 1, col = blockIdx.x * a.cols;
      row = (ct < CT / 2 ? 0 : F) + (j < a.cols && col + j < F ? col + j : col);
    } else if (MODE == SK_QKV) {
      const int half = a.D >> 1, per = half / a.cols;  // workgroups of a head
      row = (blockIdx.x / per) * a.D + (blockIdx.x % per) * a.cols + (r < a.cols ? r : r < 2 * a.cols ? r - a.cols + half : 0);
    } else {
      const int j = 16 * ct + r, col = blockIdx.x * a.cols;
      row = j < a.cols && col + j < a.N ? col + j : col;
    }
    wp[ct] = a.W + (size_t)row * a.K + 8 * kq;
  }
  const int rm = r < a.M ? r : 0;
  const bf16_t* xp = a.X + (size_t)rm * a.xs + 8 * kq;

  constexpr int SETS = PRE ? 2 : 1;
  bf16x8 wf[SETS][U][2][CT], xf[SETS][NORM ? 1 : U][2];
  auto load = [&](int set, int first) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (first + u < mine) {  // the same for all lanes
        const int k = (wave + WAVES * (first + u)) * 64;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) wf[set][u][s][ct] = ld8(wp[ct] + k + 32 * s);
          if (!NORM) xf[set][NORM ? 0 : u][s] = ld8(xp + k + 32 * s);
        }
      }
    }
  };
  load(0, 0);
  __builtin_amdgcn_sched_barrier(0);
  int rj = 0, rrow = 0;  // SK_RES: this thread's result, cols x M <= THREADS of them
  float res = 0.f;
  if (MODE == SK_RES) {
    rrow = threadIdx.x / a.cols;
    rj = threadIdx.x - rrow * a.cols;
    if (a.res) res = bf2f(a.res[(size_t)min(rrow, a.M - 1) * a.N + min((int)blockIdx.x * a.cols + rj, a.N - 1)]);
    __builtin_amdgcn_sched_barrier(0);
  }

  if (NORM) {
    if (wave < a.M) {
      float ss = 0.f;
      for (int c = lane * 8, p = 0; c < a.K; c += 512, ++p) {
        const bf16x8 h = p == 0 ? hv[0] : p == 1 ? hv[1] : p == 2 ? hv[2] : ld8(a.X + (size_t)wave * a.xs + c);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += bf2f(h[e]) * bf2f(h[e]);
      }
      const float rstd = rsqrtf(wave_sum(ss) / (float)a.K + a.eps);
      for (int c = lane * 8, p = 0; c < a.K; c += 512, ++p) {
        const bf16x8 h = p == 0 ? hv[0] : p == 1 ? hv[1] : p == 2 ? hv[2] : ld8(a.X + (size_t)wave * a.xs + c);
        const bf16x8 g = p == 0 ? gv[0] : p == 1 ? gv[1] : p == 2 ? gv[2] : ld8(a.nw + c);
        bf16x8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = f2bf(bf2f(h[e]) * rstd * (bf2f(g[e]) + (a.gemma ? 1.f : 0.f)));
        st8(xn + (size_t)wave * (a.K + 8) + c, o);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  }

  f32x4 acc[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) acc[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](int set, int first) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (first + u < mine) {
        const int k = (wave + WAVES * (first + u)) * 64;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const bf16x8 b = NORM ? ld8(xn + (size_t)rm * (a.K + 8) + k + 32 * s + 8 * kq) : xf[set][NORM ? 0 : u][s];
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
            acc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[set][u][s][ct], b, acc[ct], 0, 0, 0);
        }
      }
    }
  };
  for (int first = 0; first < mine; first += SETS * U) {
#pragma unroll
    for (int set = 0; set < SETS; ++set) {
      if (PRE) load(set ^ 1, first + (set + 1) * U);
      multiply(set, first + set * U);
      if (!PRE) load(0, first + U);
    }
  }

  // the waves' partial sums meet in LDS: [wave][tile][lane] of 4 (weight row 4 kq + i, activation row r)
  if (NORM) __syncthreads();  // in the place of the normalised rows
  f32x4* red = reinterpret_cast<f32x4*>(smem);
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) red[(wave * CT + ct) * 64 + lane] = acc[ct];
  __syncthreads();
  const float* rf = reinterpret_cast<const float*>(red);
  finish<MODE>(a, rj, rrow, res, [&](int j, int h, int m) {
    const int row = MODE == SK_QKV ? j + h * a.cols : j & 15;  // of the tile
    const int ct = MODE == SK_QKV ? 0 : (j >> 4) + h * (CT / 2);
    const int at = ct * 256 + ((row >> 2) * 16 + m) * 4 + (row & 3);
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) s += rf[w * CT * 256 + at];
    return s;
  });
}

// The packed q|k|v projection of rows that are normalised already, with bias, rotation and KV-cache write: a workgroup owns 16 RT
// rows and 8 rotated pairs over all of K, its 8 waves deal the 64-deep chunks of K among themselves, every operand goes from memory
// to the registers of the one wave that multiplies it (up to 1536 deep all of them at once), and the partial sums meet in LDS.
// What bounds it: one round trip to memory and the load path of a CU, 32 K (1 + RT) bytes a workgroup; the split-K GEMM and the row
// kernel behind it that this replaces are two launches and a round trip of fp32 slabs. Captured, cold weights, us of the two / this:
// 1536 deep to 2048 columns 9 / 16 / 24 / 32 / 48 / 64 rows 7.2 / 5.3, 7.4 / 5.8, 7.5 / 5.9, 7.5 / 6.1, 8.2 / 7.8, 8.5 / 8.2; 896 to
// 1152 9 / 48 / 96 rows 6.3 / 4.3, 7.5 / 4.8, 7.9 / 6.2; 1024 to 4096 16 / 32 rows 7.4 / 5.1, 8.5 / 7.1; 2048 to 2560 16 rows 8.6 / 7.6.
// 32 columns a workgroup or 64 rows (fewer loads of the other operand) were slower wherever one round of workgroups is enough
// (24 rows of the first: 7.4 to 8.7), and beyond that the split-K GEMM is ahead (128 rows 10.2 / 11.1). Since then without a division
// and without a wait ahead of the operands (a bias that was widened where it was loaded held them back): 12 / 24 / 48 rows of the first
// 6.00 -> 5.43, 6.38 -> 5.84, 8.22 -> 7.77.
template <int RT>
__global__ __launch_bounds__(THREADS, 4) void qkv_rows_kernel(const SKArgs a) {
  constexpr int PAIRS = 8, ITEMS = 16 * RT * PAIRS, NI = (ITEMS + THREADS - 1) / THREADS, U = 3;
  __shared__ f32x4 red[WAVES * RT * 64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, kq = lane >> 4;
  // grid: (8 XCDs, row blocks, column blocks of an XCD): a range of columns, all rows of it one after the other
  const int half = a.D >> 1, ncb = (a.N >> 1) / PAIRS;
  const int cb0 = blockIdx.x * gridDim.z + blockIdx.z, cb = min(cb0, ncb - 1), m0 = blockIdx.y * 16 * RT;
  const int head = quotient(cb, half / PAIRS, a.per_inv), d0 = (cb - head * (half / PAIRS)) * PAIRS;
  const int nchunk = a.K >> 6;
  const int mine = wave < nchunk ? (nchunk - wave + WAVES - 1) / WAVES : 0;
  const bool rot = a.do_rope && head < a.Hq + a.Hkv;

  // what the results need: on its way ahead of the operands, and not looked at before them
  int pos[NI];
  int64_t slot[NI];
  bf16_t blo[NI], bhi[NI];
  const bf16_t* bias = (a.bias ? a.bias : a.W) + head * a.D + d0;  // (without one: values that are not used)
  const int* positions = a.pos;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int idx = threadIdx.x + i * THREADS, m = min(m0 + idx / PAIRS, a.M - 1);
    pos[i] = positions[m];
    slot[i] = a.slots[m];
    blo[i] = bias[idx % PAIRS];
    bhi[i] = bias[idx % PAIRS + half];
  }
  const bf16_t* wp = a.W + (size_t)(head * a.D + d0 + (r & 7) + (r >> 3) * half) * a.K + 8 * kq;  // pair j: rows j and j + 8 of the tile
  const bf16_t* xp[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) xp[rt] = a.X + (size_t)min(m0 + rt * 16 + r, a.M - 1) * a.xs + 8 * kq;  // (rows past the last repeat it)
  __builtin_amdgcn_sched_barrier(0);

  bf16x8 wf[U][2], xf[U][2][RT];
  auto load = [&](int u, int i) __attribute__((always_inline)) {
    const int k = (wave + WAVES * i) * 64;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      wf[u][s] = ld8(wp + k + 32 * s);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) xf[u][s][rt] = ld8(xp[rt] + k + 32 * s);
    }
  };
  f32x4 acc[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) acc[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](int u) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u][s], xf[u][s][rt], acc[rt], 0, 0, 0);
  };
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (u < mine) load(u, u);
  __builtin_amdgcn_sched_barrier(0);
  float c[NI], s[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int p = max(0, min(pos[i], a.max_pos - 1)), d = d0 + (threadIdx.x + i * THREADS) % PAIRS;
    c[i] = a.cos_t[(size_t)p * half + d];
    s[i] = a.sin_t[(size_t)p * half + d];
  }
  __builtin_amdgcn_sched_barrier(0);
  int i = 0;
  for (; i + 2 * U <= mine; i += U)
#pragma unroll
    for (int u = 0; u < U; ++u) {
      multiply(u);
      __builtin_amdgcn_sched_barrier(0);
      load(u, i + U + u);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (i + u < mine) {
      multiply(u);
      if (i + U + u < mine) load(u, i + U + u);
    }
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (i + U + u < mine) multiply(u);

  // partial sums: [wave][row tile][lane] of 4 (weight row 4 kq + e, row r)
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) red[(wave * RT + rt) * 64 + lane] = acc[rt];
  __syncthreads();
  const float* rf = reinterpret_cast<const float*>(red);
#pragma unroll
  for (int n = 0; n < NI; ++n) {
    const int idx = threadIdx.x + n * THREADS, m = idx / PAIRS, j = idx % PAIRS;
    if (idx >= ITEMS || m0 + m >= a.M) continue;
    float v[2] = {0.f, 0.f};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int row = j + 8 * h, at = (m >> 4) * 256 + ((row >> 2) * 16 + (m & 15)) * 4 + (row & 3);
#pragma unroll
      for (int w = 0; w < WAVES; ++w) v[h] += rf[w * RT * 256 + at];
    }
    if (cb0 < ncb)
      put_pair(a, head, d0 + j, m0 + m, v[0], v[1], a.bias ? bf2f(blo[n]) : 0.f, a.bias ? bf2f(bhi[n]) : 0.f, rot ? c[n] : 1.f,
               rot ? s[n] : 0.f, head < a.Hq ? -1 : slot[n]);
  }
}

template <int MT, int RB, int WK, bool NORM, int MODE, bool PARTS, bool TURNS = false>
int sk_dot_as(const SKArgs& a, dim3 grid, hipStream_t st) {
  size_t lds = (size_t)WK * (MODE == SK_RES ? a.cols : 2 * a.cols) * MT * sizeof(float);
  if (PARTS) lds = (lds + 15) / 16 * 16 + (size_t)a.K * sizeof(bf16_t);
  if (lds > 64 * 1024) return -4;
  hipLaunchKernelGGL((skinny_dot_kernel<MT, RB, WK, NORM, MODE, TURNS, PARTS>), grid, dim3(THREADS), lds, st, a);
  return (int)hipGetLastError();
}

// A wave with one or two rows (o, qkv) takes sets of one: sums of rows that it does not have are not worked out.
template <int MT, int RB, int WK, bool NORM, int MODE, bool PARTS>
int sk_dot_rows(const SKArgs& a, dim3 grid, hipStream_t st) {
  if constexpr (MODE != SK_GATED)
    if ((MODE == SK_RES ? a.cols : 2 * a.cols) <= 2 * (WAVES / WK)) return sk_dot_as<MT, 1, WK, NORM, MODE, PARTS>(a, grid, st);
  return sk_dot_as<MT, RB, WK, NORM, MODE, PARTS>(a, grid, st);
}

template <int MT, int RB, bool NORM, int MODE, bool PARTS = false>
int sk_dot(const SKArgs& a, dim3 grid, hipStream_t st) {
  if constexpr (MT <= 2) {
    if (a.K <= P * 512) return sk_dot_rows<MT, RB, 1, NORM, MODE, PARTS>(a, grid, st);
    if (a.K <= 2 * P * 512) return sk_dot_rows<MT, RB, 2, NORM, MODE, PARTS>(a, grid, st);
  }
  if (a.K <= 4 * P * 512) return sk_dot_rows<MT, RB, 4, NORM, MODE, PARTS>(a, grid, st);
  if (a.K <= WAVES * P * 512) return sk_dot_rows<MT, RB, WAVES, NORM, MODE, PARTS>(a, grid, st);
  if constexpr (!NORM) return sk_dot_as<MT, RB, WAVES, NORM, MODE, PARTS, true>(a, grid, st);
  return -4;
}

template <int CT, int U, bool PRE, bool NORM, int MODE>
int sk_mfma(const SKArgs& a, int blocks, hipStream_t st) {
  const size_t sums = (size_t)WAVES * CT * 1024, rows = NORM ? (size_t)a.M * (a.K + 8) * sizeof(bf16_t) : 0;
  const size_t lds = sums > rows ? sums : rows;
  if (lds > 160 * 1024) return -4;
  if (lds > 64 * 1024)
    HIP_RET(hipFuncSetAttribute((const void*)skinny_mfma_kernel<CT, U, PRE, NORM, MODE>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
  hipLaunchKernelGGL((skinny_mfma_kernel<CT, U, PRE, NORM, MODE>), dim3(blocks), dim3(THREADS), lds, st, a);
  return (int)hipGetLastError();
}

int sk_check(const void* X, int64_t xs, const void* W, int M, int N, int K) {
  if (M < 1 || M > 8 || K < 64 || K % 64 != 0 || xs % 8 != 0 || N < 1) return -1;
  if (((uintptr_t)X | (uintptr_t)W) % 16 != 0) return -2;
  return 0;
}

constexpr int CUS = 256;

}  // namespace

// Y [M, N] = bf16(X W^T) + residual (may be null), rounded again. M <= 8, K % 64 == 0.
extern "C" int areal_skinny_residual(const void* X, int64_t xs, const void* W, const void* res, void* Y, int M, int N, int K,
                                     hipStream_t st) {
  if (int rc = sk_check(X, xs, W, M, N, K)) return rc;
  SKArgs a = {};
  a.X = (const bf16_t*)X; a.xs = xs; a.W = (const bf16_t*)W; a.res = (const bf16_t*)res; a.Y = (bf16_t*)Y;
  a.M = M; a.N = N; a.K = K;
  a.cols = (N + CUS - 1) / CUS < 16 ? (N + CUS - 1) / CUS : 16;
  const int blocks = (N + a.cols - 1) / a.cols;
  if (M == 1) return sk_dot<1, 3, false, SK_RES>(a, dim3(blocks), st);
  if (M == 2) return sk_dot<2, 3, false, SK_RES>(a, dim3(blocks), st);
  // Three rows and more: a tile of 16 weight rows holds only cols of its own, so with few of them the dot products are faster where rows
  // are long (us, 3 / 4 / 6 / 8 rows, matrix cores and dot products: 1536 columns 8960 deep, 6 a workgroup, 12.3 / 12.5 / 12.9 / 13.5 and
  // 8.5 / 8.7 / 9.8 / 10.4, 4096 deep 6.8 / 6.9 / 7.0 / 7.2 and 5.3 / 5.4 / 6.1 / 6.6, 2048 deep 4.8 / 4.7 / 5.0 / 5.1 and 4.1 / 4.2 / 4.9 / 5.2;
  // 2048 columns 6144 deep, 8 each, 10.4 / 10.6 / 9.4 / 9.8 and 7.8 / 8.0 / 9.2 / 9.4; 3584 x 3584, 14 each, 8.0 / 8.1 / 8.7 / 8.3 and 8.4 /
  // 8.6 / 10.2 / 10.7), and fewer of their values are rounded the other way than 64-bit sums (8960 deep 1e-4 and 2e-4).
  const bool deep = K > 64 * WAVES * 6;
  if (a.cols <= 8 && deep) switch (M) {
    case 3: return sk_dot<3, 3, false, SK_RES>(a, dim3(blocks), st);
    case 4: return sk_dot<4, 3, false, SK_RES>(a, dim3(blocks), st);
    case 5: return sk_dot<5, 3, false, SK_RES>(a, dim3(blocks), st);
    case 6: return sk_dot<6, 3, false, SK_RES>(a, dim3(blocks), st);
    case 7: return sk_dot<7, 3, false, SK_RES>(a, dim3(blocks), st);
    case 8: return sk_dot<8, 3, false, SK_RES>(a, dim3(blocks), st);
  }
  return deep ? sk_mfma<1, 6, true, false, SK_RES>(a, blocks, st) : sk_mfma<1, 6, false, false, SK_RES>(a, blocks, st);
}

// The same of one row of the decode attention's output, K = Hq heads of D (64, 128 or 256), that it has left as rows[0].y > 1 partial
// results from rows[0].x on, part_o [.., Hq, D] and part_ml [.., Hq, 2], or written to X.
extern "C" int areal_skinny_parts_residual(const void* X, const float* part_o, const float* part_ml, const void* rows, const void* W,
                                           const void* res, void* Y, int N, int Hq, int D, hipStream_t st) {
  if (Hq < 1 || (D != 64 && D != 128 && D != 256)) return -1;
  if (int rc = sk_check(X, 0, W, 1, N, Hq * D)) return rc;
  if ((uintptr_t)part_o % 16 != 0 || ((uintptr_t)part_ml | (uintptr_t)rows) % 8 != 0) return -2;
  SKArgs a = {};
  a.X = (const bf16_t*)X; a.W = (const bf16_t*)W; a.res = (const bf16_t*)res; a.Y = (bf16_t*)Y; a.M = 1; a.N = N; a.K = Hq * D;
  a.part_o = part_o; a.part_ml = part_ml; a.rows = (const int2*)rows; a.d_shift = D == 64 ? 6 : D == 128 ? 7 : 8;
  a.cols = (N + CUS - 1) / CUS < 16 ? (N + CUS - 1) / CUS : 16;
  return sk_dot<1, 3, false, SK_RES, true>(a, dim3((N + a.cols - 1) / a.cols), st);
}

// Y [M, F] = gate(h W_gate^T) * (h W_up^T), h = RMSNorm(X) nw, W = [gate; up] [2F, K]. K <= 8192.
extern "C" int areal_skinny_norm_gated(const void* X, int64_t xs, const void* nw, const void* W, void* Y, int M, int F, int K,
                                       float eps, int gemma, int act, hipStream_t st) {
  if (int rc = sk_check(X, xs, W, M, F, K)) return rc;
  if ((uintptr_t)nw % 16 != 0) return -3;
  SKArgs a = {};
  a.X = (const bf16_t*)X; a.xs = xs; a.nw = (const bf16_t*)nw; a.W = (const bf16_t*)W; a.Y = (bf16_t*)Y;
  a.M = M; a.N = 2 * F; a.K = K; a.eps = eps; a.gemma = gemma; a.act = act;
  int rounds = 1;
  while ((F + CUS * rounds - 1) / (CUS * rounds) > 48) ++rounds;
  a.cols = (F + CUS * rounds - 1) / (CUS * rounds);
  const int blocks = (F + a.cols - 1) / a.cols;
  if (M == 1) return sk_dot<1, 5, true, SK_GATED>(a, dim3(blocks), st);
  if (M == 2) return sk_dot<2, 5, true, SK_GATED>(a, dim3(blocks), st);
  if (a.cols <= 16) return sk_mfma<2, 3, true, true, SK_GATED>(a, blocks, st);
  if (a.cols <= 32) return sk_mfma<4, 3, false, true, SK_GATED>(a, blocks, st);
  return sk_mfma<6, 3, false, true, SK_GATED>(a, blocks, st);
}

// The packed q|k|v projection of RMSNorm(X) nw with bias, rotation and KV-cache write; returns the rotated q in Y
// [M, Hq, D]. D a multiple of 16, K <= 8192.
extern "C" int areal_skinny_norm_qkv(const void* X, int64_t xs, const void* nw, const void* W, const void* bias,
                                     const int* pos, const int64_t* slots, const float* cos_t, const float* sin_t, void* Y,
                                     void* kcache, void* vcache, int M, int K, int Hq, int Hkv, int D, int max_pos,
                                     int do_rope, float eps, int gemma, int fp8, hipStream_t st) {
  const int N = (Hq + 2 * Hkv) * D;
  if (int rc = sk_check(X, xs, W, M, N, K)) return rc;
  if (D % 16 != 0 || (uintptr_t)nw % 16 != 0) return -3;
  SKArgs a = {};
  a.X = (const bf16_t*)X; a.xs = xs; a.nw = (const bf16_t*)nw; a.W = (const bf16_t*)W; a.bias = (const bf16_t*)bias;
  a.Y = (bf16_t*)Y; a.M = M; a.N = N; a.K = K; a.eps = eps; a.gemma = gemma; a.pos = pos; a.slots = slots; a.cos_t = cos_t;
  a.sin_t = sin_t; a.kcache = kcache; a.vcache = vcache; a.Hq = Hq; a.Hkv = Hkv; a.D = D; a.max_pos = max_pos;
  a.do_rope = do_rope; a.fp8 = fp8;
  a.cols = N / 8 <= CUS ? 4 : 8;  // rotated pairs of a workgroup
  const int blocks = N / (2 * a.cols);
  const dim3 of_head(D / 2 / a.cols, Hq + 2 * Hkv);
  if (M == 1) return sk_dot<1, 3, true, SK_QKV>(a, of_head, st);
  if (M == 2) return sk_dot<2, 3, true, SK_QKV>(a, of_head, st);
  return sk_mfma<1, 3, true, true, SK_QKV>(a, blocks, st);
}

// The same of rows that are normalised already, any number of them: 16 rt rows (rt 1 or 2) and 8 pairs a workgroup. D a multiple of 16.
extern "C" int areal_qkv_rows(const void* X, int64_t xs, const void* W, const void* bias, const int* pos, const int64_t* slots,
                              const float* cos_t, const float* sin_t, void* Y, void* kcache, void* vcache, int M, int K, int Hq,
                              int Hkv, int D, int max_pos, int do_rope, int fp8, int rt, hipStream_t st) {
  if (M < 1 || K < 64 || K % 64 != 0 || xs % 8 != 0 || D < 16 || D % 16 != 0 || (rt != 1 && rt != 2)) return -1;
  if (((uintptr_t)X | (uintptr_t)W) % 16 != 0) return -2;
  SKArgs a = {};
  a.X = (const bf16_t*)X; a.xs = xs; a.W = (const bf16_t*)W; a.bias = (const bf16_t*)bias; a.Y = (bf16_t*)Y; a.M = M;
  a.N = (Hq + 2 * Hkv) * D; a.K = K; a.pos = pos; a.slots = slots; a.cos_t = cos_t; a.sin_t = sin_t; a.kcache = kcache;
  a.vcache = vcache; a.Hq = Hq; a.Hkv = Hkv; a.D = D; a.max_pos = max_pos; a.do_rope = do_rope; a.fp8 = fp8;
  if (!do_rope) {  // no angles are used: what is read in their place, D / 2 floats, is the weight's first bytes, whatever the tables hold
    a.cos_t = a.sin_t = (const float*)W;
    a.max_pos = 1;
  }
  const int cols = a.N / 16, per = D / 16, most = 65535 * 16 * rt;  // rows of a launch
  if ((cols + 7) / 8 > 65535) return -1;
  a.per_inv = reciprocal(cols, per);
  for (int m = 0; m < M; m += most) {
    a.M = M - m < most ? M - m : most;
    const dim3 grid(8, (a.M + 16 * rt - 1) / (16 * rt), (cols + 7) / 8);
    if (rt == 1) hipLaunchKernelGGL(qkv_rows_kernel<1>, grid, dim3(THREADS), 0, st, a);
    else hipLaunchKernelGGL(qkv_rows_kernel<2>, grid, dim3(THREADS), 0, st, a);
    a.X += (size_t)most * xs; a.Y += (size_t)most * Hq * D; a.pos += most; a.slots += most;
  }
  return (int)hipGetLastError();
}
