// Variable-length causal flash attention, forward and backward, for gfx950 (CDNA4).
//
// Owns what the reference borrows from flash-attn 2 (flash_attn_varlen_func at
// realhf/impl/model/modules/attn.py:289 and HF attn_implementation=flash_attention_2 via
// areal/engine/base_hf_engine.py:291-406): packed [T, H, D] q/k/v with cu_seqlens, GQA,
// causal masking aligned to the bottom-right corner when q and k lengths differ.
//
// Both kernels are built on v_mfma_f32_32x32x16_bf16 and arrange every product so that an
// accumulator tile feeds the next MFMA as an operand without leaving registers:
//   forward : S^T = K.Q^T (key in the accumulator rows, query on the lane) so the softmax
//             row statistics are lane-local; O^T += V^T.P^T takes P from the accumulator
//             registers as the B operand; V^T fragments come from ds_read_b64_tr_b16.
//   backward: S = Q.K^T and dP = dO.V^T keep the key on the lane, so P and dS are already the B operands of
//             dV^T += dO^T.P and dK^T += Q^T.dS; a second, query-major kernel (forward-shaped) recomputes S and dP for
//             dQ^T += K^T.dS^T.
// LDS tiles use 256-byte rows with the 16-byte-chunk XOR swizzle
//   off(row, ch) = 256*row + 16*(ch ^ (((row&3)<<2) | ((row>>2)&3)))
// which is conflict-free for both ds_read_b128 row reads and transposed reads.
#include <type_traits>

#include "flash_tiles.hpp"

// =====================================================================================
// Forward. 1-D grid over (q-tile rank, sequence, head). block: 256 threads = 4 waves x 32 q rows.
// KV tile = 64 keys. D = 128.
//
// What bounds it: a wave's 32 x 64 scores take 1024 cycles of matrix pipe per tile and about as much of the vector pipe
// (32 exponentials and eight more operations each per lane), so the two have to overlap: two workgroups a CU (two waves a
// SIMD, 228 registers each) that run apart:
//   * tiles that no query of the wave may miss a key of run without mask code, tiles it sees no key of are skipped;
//   * K and V tiles come by LDS-DMA into two buffers: no staging registers, one barrier a tile.
// A row's scores are scaled (rounded once), its maximum follows every tile and the exponential takes the difference: what
// comes out of a row depends on that row alone, bit for bit, whatever else is packed beside it. (Folding the scale into the
// exponential's argument and rescaling only when some row of the wave has grown by more than 2^8 takes 5-7 % less time, but
// then the rows of a wave decide on each other's rounding, and a training pass over 32768 tokens and 7 layers moves the final
// norm's gradient, elements of some 300 times the overall rms, by 0.7 %.)
// Measured (12 query heads on 2 key heads), register-staged tiles, one workgroup's waves in step -> this: 25 sequences of 1133
// tokens 177 -> 151 us, 2 of 300 15.0 -> 11.5 us, 24576 tokens 2.13 -> 1.86 ms (873 -> 998 TFLOP/s); 3 x 8192 (28 on 4
// heads) 1.94 -> 1.62 ms; since the next tile's DMA is no longer waited for at once (dma16) 143 us, 1.78 ms (1030 TFLOP/s), 1.60 ms.
// =====================================================================================
__global__ __launch_bounds__(256, 2) void flash_fwd_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k, const bf16_t* __restrict__ v,
    bf16_t* __restrict__ o, float* __restrict__ lse, const int* __restrict__ cu_q,
    const int* __restrict__ cu_k, int64_t q_stride, int64_t k_stride, int64_t v_stride,
    int64_t o_stride, int Hq, int Hkv, int nbatch, int total_q, float scale_log2, int causal) {
  constexpr int D = 128;
  __shared__ __attribute__((aligned(16))) char smem[2 * 2 * 64 * 256];  // [buffer][K, V]
  // 1-D grid, query-tile rank first: rank 0 is the LAST (heaviest under causal masking) tile of every
  // (sequence, head), so heavy workgroups of all sequences start first and light ones fill the tail.
  // XCD placement: consecutive workgroup ids go round-robin over the 8 XCDs, each with its own L2. Inside
  // a rank the slot of the (sequence, kv head) group runs fastest over an extent padded to a multiple of 8,
  // and group g sits in slot (g + rank) mod extent, so id % 8 == (g + rank) % 8: all query heads that read
  // the K/V of one group for one query tile run on the same XCD and share those tiles in its L2, while the
  // rotation by rank spreads a group's query tiles - and with them the padding slots and any remainder
  // of the group count modulo 8 - evenly over the XCDs (without it a single long sequence with two kv
  // heads would keep six of the eight XCDs idle).
  const int G = Hq / Hkv;
  const int n_g = Hkv * nbatch, n_g_pad = (n_g + 7) & ~7;
  const int per_rank = G * n_g_pad;
  const int rank = blockIdx.x / per_rank, rem = blockIdx.x - rank * per_rank;
  const int hj = rem / n_g_pad, slot = rem - hj * n_g_pad;
  int g = slot - rank % n_g_pad;
  g += g < 0 ? n_g_pad : 0;
  if (g >= n_g) return;
  const int b = g / Hkv, head = (g - b * Hkv) * G + hj;
  const int q_beg = cu_q[b], q_len = cu_q[b + 1] - q_beg;
  const int k_beg = cu_k[b], k_len = cu_k[b + 1] - k_beg;
  const int ntile_q = (q_len + 127) / 128;
  if (rank >= ntile_q) return;
  const int qt = ntile_q - 1 - rank;
  const int kvh = head / (Hq / Hkv);
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 31, hf = lane >> 5, gl = lane & 15, grp = lane >> 4;
  const int shift = k_len - q_len;  // bottom-right aligned causal mask

  const int q0 = qt * 128 + wid * 32;  // first q row of this wave (within the sequence)
  const int my_q = q0 + r;
  const int my_q_c = my_q < q_len ? my_q : q_len - 1;
  // Q^T as the B operand: lane (r, hf) holds Q[r][16ks + 8hf + j]
  bf16x8 qf[8];
  {
    const bf16_t* qp = q + (size_t)(q_beg + my_q_c) * q_stride + (size_t)head * D + hf * 8;
#pragma unroll
    for (int s = 0; s < 8; ++s) qf[s] = ld8(qp + s * 16);
  }
  f32x16 oacc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) oacc[i][j] = 0.f;
  float m = -INFINITY, l = 0.f;  // maximum of the scaled scores; sum of this lane's keys

  // number of kv tiles this block needs (the whole block walks the same range)
  int k_hi = k_len;
  if (causal) {
    const int last_q = min(q_len, qt * 128 + 128) - 1;
    k_hi = min(k_len, last_q + shift + 1);
  }
  const int ntile_k = k_hi > 0 ? (k_hi + 63) / 64 : 0;
  const bf16_t* kbase_p = k + (size_t)k_beg * k_stride + (size_t)kvh * D;
  const bf16_t* vbase_p = v + (size_t)k_beg * v_stride + (size_t)kvh * D;
  const FragOffsets fo(lane);
  unsigned koff[4], voff[4];
  dma_offsets(koff, wid, lane, k_stride);
  dma_offsets(voff, wid, lane, v_stride);
  auto issue = [&](int t) {
    char* buf = smem + (t & 1) * 32768;
    dma_tile(kbase_p + (size_t)t * 64 * k_stride, koff, k_stride, k_len - t * 64, buf, wid, lane);
    dma_tile(vbase_p + (size_t)t * 64 * v_stride, voff, v_stride, k_len - t * 64, buf + 16384, wid, lane);
  };

  auto step = [&](int t, auto masked) {
    const char* ks = smem + (t & 1) * 32768;
    const char* vs = ks + 16384;
    const int kbase = t * 64;
    // ---- S^T = K . Q^T : two 32-key blocks
    f32x16 sacc[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
      // fragments are read four at a time ahead of the MFMAs that use them, so that an MFMA waits for a
      // read issued four instructions earlier instead of for the one just before it
      for (int s0 = 0; s0 < 8; s0 += 4) {
        bf16x8 kf[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) kf[s] = *reinterpret_cast<const bf16x8*>(ks + (fo.row(s0 + s) + 8192 * kb));
        __builtin_amdgcn_sched_barrier(0);  // keep the scheduler from sinking the reads back to their uses
#pragma unroll
        for (int s = 0; s < 4; ++s) sacc[kb] = mfma32(kf[s], qf[s0 + s], s0 + s ? sacc[kb] : f32x16{});
      }
    }
    // ---- online softmax; lane holds q row `my_q`, keys (reg&3)+8(reg>>2)+4hf of each block
    float mx = -INFINITY, ls = 0.f;
    bf16x8 pf[4];
    {
#pragma clang fp contract(off)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          sacc[kb][j] *= scale_log2;
          if (decltype(masked)::value) {
            const int key = kbase + 32 * kb + (j & 3) + 8 * (j >> 2) + 4 * hf;
            sacc[kb][j] = key >= k_len || (causal && key > my_q + shift) ? -INFINITY : sacc[kb][j];
          }
          mx = fmaxf(mx, sacc[kb][j]);
        }
      mx = max_xor32(mx);
      const float mn = fmaxf(m, mx);
      const float alpha = mn == -INFINITY ? 1.f : fast_exp2(m - mn);  // m = -inf -> 0
      m = mn;
      if (__any(m == -INFINITY)) {  // rows that have seen no key yet: probabilities of zero
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int j = 0; j < 16; ++j) sacc[kb][j] = m == -INFINITY ? -INFINITY : sacc[kb][j];
      }
      const float ms = m == -INFINITY ? 0.f : m;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const float pr = fast_exp2(sacc[kb][j] - ms);
          ls += pr;
          pf[2 * kb + (j >> 3)][j & 7] = f2bf(pr);
        }
      l = __builtin_fmaf(l, alpha, ls);
      if (__any(alpha != 1.f)) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 16; ++j) oacc[i][j] *= alpha;
      }
    }
    // ---- O^T[d, q] += V^T[d, keys] . P^T[keys, q]
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      // group `grp`: rows = keys 16s + 4hf (+8), cols = d 32db + 16(grp&1); all eight transposed reads of
      // a key slab are issued before its four MFMAs
      bf16x4 a0[4], a1[4];
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        a0[db] = tr_load(vs + (fo.tr0(db) + 4096 * s));
        a1[db] = tr_load(vs + (fo.tr1(db) + 4096 * s));
      }
#pragma unroll
      for (int db = 0; db < 4; ++db) oacc[db] = mfma32(cat4(a0[db], a1[db]), pf[s], oacc[db]);
    }
  };

  // tiles of which no query of this wave may miss a key, then the others, of which those behind the wave's last query hold
  // none (every wave passes every barrier)
  int n_full = k_len / 64;
  if (causal) n_full = min(n_full, max(0, (q0 + shift + 1) / 64));
  n_full = min(n_full, ntile_k);
  if (ntile_k > 0) issue(0);
  dma_pin(qf);
  int t = 0;
  for (; t < n_full; ++t) {
    dma_arrive();
    if (t + 1 < ntile_k) issue(t + 1);
    step(t, std::false_type{});
  }
  for (; t < ntile_k; ++t) {
    dma_arrive();
    if (t + 1 < ntile_k) issue(t + 1);
    if (!causal || t * 64 <= q0 + 31 + shift) step(t, std::true_type{});
  }
  // ---- epilogue
  l = sum_xor32(l);
  const float inv_l = l > 0.f ? 1.f / l : 0.f;
  if (my_q < q_len) {
    bf16_t* op = o + (size_t)(q_beg + my_q) * o_stride + (size_t)head * D;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        bf16x4 w;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = f2bf(oacc[db][4 * g + j] * inv_l);
        *reinterpret_cast<bf16x4*>(op + 32 * db + 8 * g + 4 * hf) = w;
      }
    if (hf == 0 && lse) {
#pragma clang fp contract(off)
      lse[(size_t)head * total_q + q_beg + my_q] =
          (l > 0.f) ? (m * 0.6931471805599453f + __logf(l)) : -INFINITY;
    }
  }
}

// head size 256: flash_attn_d256.hip
extern "C" int areal_flash_fwd_d256(const void* q, const void* k, const void* v, void* o, float* lse,
                                    const int* cu_q, const int* cu_k, int B, int max_q, int total_q, int Hq, int Hkv,
                                    int64_t q_stride, int64_t k_stride, int64_t v_stride, int64_t o_stride,
                                    float softmax_scale, int causal, hipStream_t st);
extern "C" int areal_flash_bwd_d256(const void* q, const void* k, const void* v, const void* o, const void* d_o,
                                    const float* lse, float* delta, void* dq, void* dk, void* dv, const int* cu_q,
                                    const int* cu_k, int B, int max_k, int total_q, int64_t total_k, int Hq, int Hkv,
                                    int64_t q_stride, int64_t k_stride, int64_t v_stride, int64_t o_stride, int64_t do_stride,
                                    int64_t dq_stride, int64_t dk_stride, int64_t dv_stride, float softmax_scale,
                                    int causal, hipStream_t st);

extern "C" int areal_flash_fwd(const void* q, const void* k, const void* v, void* o, float* lse,
                               const int* cu_q, const int* cu_k, int B, int max_q, int total_q,
                               int Hq, int Hkv, int D, int64_t q_stride, int64_t k_stride,
                               int64_t v_stride, int64_t o_stride, float softmax_scale, int causal,
                               hipStream_t st) {
  if (B == 0 || max_q == 0) return 0;
  if (D != 128 && D != 256) return -1;
  if (Hq % Hkv != 0) return -2;
  if ((q_stride | k_stride | v_stride | o_stride) % 8 != 0) return -3;
  if (k_stride > FLASH_MAX_STRIDE || v_stride > FLASH_MAX_STRIDE) return -5;
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)o) % 16 != 0) return -4;
  if (D == 256)
    return areal_flash_fwd_d256(q, k, v, o, lse, cu_q, cu_k, B, max_q, total_q, Hq, Hkv, q_stride, k_stride, v_stride,
                                o_stride, softmax_scale, causal, st);
  const int n_g_pad = (Hkv * B + 7) & ~7;  // see the XCD placement note in the kernel
  dim3 grid((unsigned)(((max_q + 127) / 128) * (Hq / Hkv) * n_g_pad)), block(256);
  hipLaunchKernelGGL(flash_fwd_kernel, grid, block, 0, st, (const bf16_t*)q, (const bf16_t*)k,
                     (const bf16_t*)v, (bf16_t*)o, lse, cu_q, cu_k, q_stride, k_stride, v_stride,
                     o_stride, Hq, Hkv, B, total_q, softmax_scale * 1.4426950408889634f, causal);
  return (int)hipGetLastError();
}

// =====================================================================================
// Backward.
//  pre : delta[h, t] = sum_d dO[t, h, d] * O[t, h, d], and the log-sum-exp in base 2; gradients of rows of no sequence
//  dkv : workgroups of 128 keys sweep the query slices that see them
//  dq  : workgroups of 128 queries walk their keys
// Seven products instead of the five that one kernel needs, but nothing is handed over: with dQ added up by fp32 atomics
// (one kernel, 132 KiB of registers and 81 KiB of LDS a workgroup, one wave a SIMD) the same batches took longer at every
// length. Forward + backward, 12 query heads on 2 key heads unless said, one kernel up to 2048 keys and two one-wave kernels
// above -> these:
//   25 x ~1133 tokens 857 -> 621 us (backward alone), 16 x 200-1216 (32 on 4 heads) 1100 -> 670 us,
//   3 x 8192 (28 on 4 heads) 8.75 -> 5.10 ms (708 TFLOP/s), 24576 10.8 -> 6.2 ms (431 -> 745 TFLOP/s).
// =====================================================================================
__global__ __launch_bounds__(256) void flash_bwd_delta_kernel(
    const bf16_t* __restrict__ o, const bf16_t* __restrict__ d_o, const float* __restrict__ lse,
    float* __restrict__ delta, int64_t o_stride, int64_t do_stride, int Hq, int total_q, const FlashGrads grads) {
  constexpr int D = 128;
  // 16 lanes per (token, head)
  const int64_t idx = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 4;
  const int sub = threadIdx.x & 15;
  const int64_t t = idx / Hq;
  const int h = (int)(idx % Hq);
  flash_zero_uncovered(grads, t, h, D, sub * 8);
  if (t >= total_q) return;
  bf16x8 a = ld8(o + t * o_stride + (size_t)h * D + sub * 8);
  bf16x8 bb = ld8(d_o + t * do_stride + (size_t)h * D + sub * 8);
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) s += bf2f(a[j]) * bf2f(bb[j]);
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if (sub == 0) {  // [0]: delta, [1]: the log-sum-exp in base 2
    delta[(size_t)h * total_q + t] = s;
    delta[(size_t)(Hq + h) * total_q + t] = lse[(size_t)h * total_q + t] * 1.4426950408889634f;
  }
}

// dQ on its own, one workgroup per 128-row query tile (the grid and XCD placement of the forward): S and dP are computed a
// second time, and nothing crosses workgroups. Same operand arrangement as the forward: S^T = K.Q^T and dP^T = V.dO^T keep
// the query on the lane (lse and delta are per-lane scalars), dS^T comes out of the accumulators as the B operand of
// dQ^T += K^T.dS^T, K^T fragments are transposed LDS reads. dQ is written once, in bf16, with the softmax scale applied.
// Staging, tile walk and what bounds it as in the forward; two workgroups a CU.
__global__ __launch_bounds__(256, 2) void flash_bwd_dq_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k, const bf16_t* __restrict__ v,
    const bf16_t* __restrict__ d_o, const float* __restrict__ delta, bf16_t* __restrict__ dq,
    const int* __restrict__ cu_q, const int* __restrict__ cu_k, int64_t q_stride, int64_t k_stride, int64_t v_stride,
    int64_t do_stride, int64_t dq_stride, int Hq, int Hkv, int nbatch, int total_q, float softmax_scale, int causal) {
  constexpr int D = 128;
  __shared__ __attribute__((aligned(16))) char smem[2 * 2 * 64 * 256];  // [buffer][K, V]
  const int G = Hq / Hkv;
  const int n_g = Hkv * nbatch, n_g_pad = (n_g + 7) & ~7;
  const int per_rank = G * n_g_pad;
  const int rank = blockIdx.x / per_rank, rem = blockIdx.x - rank * per_rank;
  const int hj = rem / n_g_pad, slot = rem - hj * n_g_pad;
  int g = slot - rank % n_g_pad;
  g += g < 0 ? n_g_pad : 0;
  if (g >= n_g) return;
  const int b = g / Hkv, head = (g - b * Hkv) * G + hj;
  const int q_beg = cu_q[b], q_len = cu_q[b + 1] - q_beg;
  const int k_beg = cu_k[b], k_len = cu_k[b + 1] - k_beg;
  const int ntile_q = (q_len + 127) / 128;
  if (rank >= ntile_q) return;
  const int qt = ntile_q - 1 - rank;
  const int kvh = head / G;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 31, hf = lane >> 5;
  const int shift = k_len - q_len;
  const float scale_log2 = softmax_scale * 1.4426950408889634f;


  const int q0 = qt * 128 + wid * 32;
  const int my_q = q0 + r;
  const bool q_ok = my_q < q_len;
  const int my_q_c = q_ok ? my_q : q_len - 1;
  bf16x8 qf[8], dof[8];
  {
    const bf16_t* qp = q + (size_t)(q_beg + my_q_c) * q_stride + (size_t)head * D + hf * 8;
    const bf16_t* dp = d_o + (size_t)(q_beg + my_q_c) * do_stride + (size_t)head * D + hf * 8;
#pragma unroll
    for (int s = 0; s < 8; ++s) { qf[s] = ld8(qp + s * 16); dof[s] = ld8(dp + s * 16); }
  }
  // rows past the end: lse = +inf makes every probability zero
  float lse2 = q_ok ? delta[(size_t)(Hq + head) * total_q + q_beg + my_q] : INFINITY;
  float dlt = q_ok ? delta[(size_t)head * total_q + q_beg + my_q] : 0.f;
  f32x16 dqacc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) dqacc[i][j] = 0.f;

  int k_hi = k_len;
  if (causal) {
    const int last_q = min(q_len, qt * 128 + 128) - 1;
    k_hi = min(k_len, last_q + shift + 1);
  }
  const int ntile_k = k_hi > 0 ? (k_hi + 63) / 64 : 0;
  const bf16_t* kbase_p = k + (size_t)k_beg * k_stride + (size_t)kvh * D;
  const bf16_t* vbase_p = v + (size_t)k_beg * v_stride + (size_t)kvh * D;
  const FragOffsets fo(lane);
  unsigned koff[4], voff[4];
  dma_offsets(koff, wid, lane, k_stride);
  dma_offsets(voff, wid, lane, v_stride);
  auto issue = [&](int t) {
    char* buf = smem + (t & 1) * 32768;
    dma_tile(kbase_p + (size_t)t * 64 * k_stride, koff, k_stride, k_len - t * 64, buf, wid, lane);
    dma_tile(vbase_p + (size_t)t * 64 * v_stride, voff, v_stride, k_len - t * 64, buf + 16384, wid, lane);
  };
  auto step = [&](int t, auto masked) {
    const char* ks = smem + (t & 1) * 32768;
    const char* vs = ks + 16384;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      // ---- S^T = K.Q^T and dP^T = V.dO^T for one block of 32 keys
      f32x16 sacc, pacc;
#pragma unroll
      for (int s0 = 0; s0 < 8; s0 += 2) {
        bf16x8 kf[2], vf[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          kf[s] = *reinterpret_cast<const bf16x8*>(ks + (fo.row(s0 + s) + 8192 * kb));
          vf[s] = *reinterpret_cast<const bf16x8*>(vs + (fo.row(s0 + s) + 8192 * kb));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          sacc = mfma32(kf[s], qf[s0 + s], s0 + s ? sacc : f32x16{});
          pacc = mfma32(vf[s], dof[s0 + s], s0 + s ? pacc : f32x16{});
        }
      }
      // ---- P^T = exp2(S^T c - lse), dS^T = P^T (dP^T - delta); lane = q row, reg -> key
      bf16x8 dsf[2];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        float pr = fast_exp2(__builtin_fmaf(sacc[j], scale_log2, -lse2));
        if (decltype(masked)::value) {
          const int key = t * 64 + 32 * kb + (j & 3) + 8 * (j >> 2) + 4 * hf;
          if (key >= k_len || (causal && key > my_q + shift)) pr = 0.f;
        }
        dsf[j >> 3][j & 7] = f2bf(pr * (pacc[j] - dlt));
      }
      // ---- dQ^T[d, q] += K^T[d, keys] . dS^T[keys, q]
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        bf16x4 a0[4], a1[4];
#pragma unroll
        for (int db = 0; db < 4; ++db) {
          a0[db] = tr_load(ks + (fo.tr0(db) + 4096 * (2 * kb + s)));
          a1[db] = tr_load(ks + (fo.tr1(db) + 4096 * (2 * kb + s)));
        }
#pragma unroll
        for (int db = 0; db < 4; ++db) dqacc[db] = mfma32(cat4(a0[db], a1[db]), dsf[s], dqacc[db]);
      }
    }
  };
  int n_full = k_len / 64;
  if (causal) n_full = min(n_full, max(0, (q0 + shift + 1) / 64));
  n_full = min(n_full, ntile_k);
  if (ntile_k > 0) issue(0);
  dma_pin(qf);
  dma_pin(dof);
  asm volatile("" : "+v"(lse2), "+v"(dlt));
  int t = 0;
  for (; t < n_full; ++t) {
    dma_arrive();
    if (t + 1 < ntile_k) issue(t + 1);
    step(t, std::false_type{});
  }
  for (; t < ntile_k; ++t) {
    dma_arrive();
    if (t + 1 < ntile_k) issue(t + 1);
    if (!causal || t * 64 <= q0 + 31 + shift) step(t, std::true_type{});
  }
  if (q_ok) {
    bf16_t* op = dq + (size_t)(q_beg + my_q) * dq_stride + (size_t)head * D;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        bf16x4 w;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = f2bf(dqacc[db][4 * g4 + j] * softmax_scale);
        *reinterpret_cast<bf16x4*>(op + 32 * db + 8 * g4 + 4 * hf) = w;
      }
  }
}

// dK and dV: one workgroup per 128 keys of a key head and `hs` of its query heads, 4 waves x 32 keys. A wave keeps its K
// fragments and the dK^T / dV^T accumulators in registers and sweeps 32-row query slices; V fragments are read from LDS, so
// that two workgroups fit a CU (256 registers a lane) and one's exponentials run under the other's matrix products.
//   S = Q.K^T and dP = dO.V^T keep the key on the lane: P and dS are already the B operands of dV^T += dO^T.P and
//   dK^T += Q^T.dS. Q and dO slices come by LDS-DMA into two buffers, one barrier a slice. Keys past the end only reach
//   columns that are not stored; query rows past the end have lse = +inf.
// With several workgroups a key block (parts > 1: part p takes query heads p hs ...) the sums go to fp32 buffers
// part[p][dK, dV][token, key head, D] that flash_bwd_sum_kernel adds in the order of p.
__global__ __launch_bounds__(256, 2) void flash_bwd_dkv_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k, const bf16_t* __restrict__ v,
    const bf16_t* __restrict__ d_o, const float* __restrict__ delta, bf16_t* __restrict__ dk, bf16_t* __restrict__ dv,
    float* __restrict__ part, const int* __restrict__ cu_q, const int* __restrict__ cu_k, int64_t q_stride,
    int64_t k_stride, int64_t v_stride, int64_t do_stride, int64_t dk_stride, int64_t dv_stride, int Hq, int Hkv,
    int nbatch, int total_q, int64_t total_k, int parts, int hs, float softmax_scale, int causal) {
  constexpr int D = 128;
  // V tile [128][256 B] | two buffers of Q [32][256 B], dO [32][256 B] | two of lse2 [32], delta [32]
  __shared__ __attribute__((aligned(16))) char smem[128 * 256 + 2 * 2 * 32 * 256 + 2 * 2 * 32 * 4];
  char* vs = smem;
  char* qds = smem + 128 * 256;
  float* rc = reinterpret_cast<float*>(qds + 2 * 2 * 32 * 256);

  // 1-D grid ordered by key block first: under causal masking the work of a workgroup falls with its key-block index, so
  // the heaviest workgroups of ALL sequences are dispatched first and the light ones fill the tail.
  const int n_bh = Hkv * nbatch * parts;
  const int kblk = blockIdx.x / n_bh;
  int rem = blockIdx.x - kblk * n_bh;
  const int pt = rem % parts;
  rem /= parts;
  const int b = rem / Hkv, kvh = rem - b * Hkv;
  const int q_beg = cu_q[b], q_len = cu_q[b + 1] - q_beg;
  const int k_beg = cu_k[b], k_len = cu_k[b + 1] - k_beg;
  const int kb0 = kblk * 128;
  if (kb0 >= k_len) return;
  const int G = Hq / Hkv;
  const int h0 = kvh * G + pt * hs, nh = min(hs, G - pt * hs);
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 31, hf = lane >> 5;
  const int shift = k_len - q_len;
  const float scale_log2 = softmax_scale * 1.4426950408889634f;

  const int kw0 = kb0 + 32 * wid;  // this wave's first key
  const int my_key = kw0 + r;
  bf16x8 kf[8];
  {
    const int my_key_c = my_key < k_len ? my_key : k_len - 1;
    const bf16_t* kp = k + (size_t)(k_beg + my_key_c) * k_stride + (size_t)kvh * D + hf * 8;
#pragma unroll
    for (int s = 0; s < 8; ++s) kf[s] = ld8(kp + s * 16);
  }
  {
    unsigned voff[4];
    dma_offsets(voff, wid, lane, v_stride);
#pragma unroll
    for (int half = 0; half < 2; ++half)
      if (kb0 + 64 * half < k_len)
        dma_tile(v + (size_t)(k_beg + kb0 + 64 * half) * v_stride + (size_t)kvh * D, voff, v_stride,
                 k_len - kb0 - 64 * half, vs + 16384 * half, wid, lane);
  }
  f32x16 dkacc[4], dvacc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) { dkacc[i][j] = 0.f; dvacc[i][j] = 0.f; }

  // query slices that can see this key block: every head's slices first .. last, walked as one flat sequence
  int first = 0;
  if (causal && kb0 - shift > 0) first = (kb0 - shift) / 32;
  const int nslice = max(0, (q_len + 31) / 32 - first);
  // slices of a head behind which the wave's keys are all visible (before: the diagonal)
  int n_diag = 0;
  if (causal) n_diag = min(nslice, max(0, (kw0 + 31 - shift + 31) / 32 - first));
  const FragOffsets fo(lane);
  unsigned qoff[2], dooff[2];
  dma_offsets32(qoff, wid, lane, q_stride);
  dma_offsets32(dooff, wid, lane, do_stride);
  const int nwork = nh > 0 ? nh * nslice : 0;
  float rc_next = 0.f;  // wave 0: lane -> lse2 (first half) or delta of the next slice's rows
  bool rc_ok = false;   // a row of the sequence
  int it = 0, n_head = h0, n_slice = 0;  // issued so far; the next slice's head and index
  auto issue = [&]() {
    char* buf = qds + (it & 1) * 16384;
    const int qs0 = (first + n_slice) * 32;
    dma_tile32(q + (size_t)(q_beg + qs0) * q_stride + (size_t)n_head * D, qoff, q_stride, q_len - qs0, buf, wid, lane);
    dma_tile32(d_o + (size_t)(q_beg + qs0) * do_stride + (size_t)n_head * D, dooff, do_stride, q_len - qs0, buf + 8192, wid,
               lane);
    if (wid == 0) {
      const int qi = qs0 + r;
      rc_next = delta[(size_t)((hf ? 0 : Hq) + n_head) * total_q + q_beg + (qi < q_len ? qi : q_len - 1)];
      rc_ok = qi < q_len;  // (chosen by when the value is stored: a choice here would wait for it, and for the slice)
    }
    if (++n_slice == nslice) { n_slice = 0; ++n_head; }
  };
  // slice `it` is complete in LDS; the one after it is on its way
  auto advance = [&]() {
    if (wid == 0) rc[(it & 1) * 64 + lane] = rc_ok ? rc_next : hf ? 0.f : INFINITY;  // waits for the value, and with it for the slice's DMA
    dma_arrive();
    ++it;
    if (it < nwork) issue();
  };
  auto step = [&](int slice, auto masked) {
    const int cur = it - 1;
    const char* qs = qds + (cur & 1) * 16384;
    const char* dos = qs + 8192;
    const float* rcs = rc + (cur & 1) * 64;
    const int qu = (first + slice) * 32;
    // ---- S = Q.K^T, dP = dO.V^T (rows = q in registers, col = key on the lane). Fragments are requested ahead of the products in
    // front of theirs, as many as there are registers for (backward pass, us, read next to their use / so: 24576 tokens, 12 heads on 2,
    // 5723 / 5617, 16384, 32 on 4, 6879 / 6707; the same in the two other kernels gives nothing).
    f32x16 sacc, pacc;
    bf16x8 qa[2][2], da[2], vf[2];
    auto read_q = [&](int g) __attribute__((always_inline)) {
#pragma unroll
      for (int s = 0; s < 2; ++s) qa[g & 1][s] = *reinterpret_cast<const bf16x8*>(qs + fo.row(2 * g + s));
    };
    auto read_d = [&](int s) __attribute__((always_inline)) {
      da[s & 1] = *reinterpret_cast<const bf16x8*>(dos + fo.row(s));
      vf[s & 1] = *reinterpret_cast<const bf16x8*>(vs + (fo.row(s) + 8192 * wid));
    };
    read_q(0);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (g < 3)
        read_q(g + 1);
      else
        read_d(0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < 2; ++s) sacc = mfma32(qa[g & 1][s], kf[2 * g + s], g + s ? sacc : f32x16{});
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      if (s < 7) read_d(s + 1);
      __builtin_amdgcn_sched_barrier(0);
      pacc = mfma32(da[s & 1], vf[s & 1], s ? pacc : f32x16{});
    }
    bf16x4 d0[2], d1[2], q0[2], q1[2];
    auto read_t = [&](int i) __attribute__((always_inline)) {
      const int s = i >> 2, db = i & 3;
      d0[i & 1] = tr_load(dos + (fo.tr0(db) + 4096 * s));
      d1[i & 1] = tr_load(dos + (fo.tr1(db) + 4096 * s));
      q0[i & 1] = tr_load(qs + (fo.tr0(db) + 4096 * s));
      q1[i & 1] = tr_load(qs + (fo.tr1(db) + 4096 * s));
    };
    read_t(0);
    // ---- P = exp2(S c - lse), dS = P (dP - delta)
    bf16x8 pfr[2], dsfr[2];
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const f32x4 l4 = *reinterpret_cast<const f32x4*>(rcs + 8 * g4 + 4 * hf);
      const f32x4 d4 = *reinterpret_cast<const f32x4*>(rcs + 32 + 8 * g4 + 4 * hf);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int reg = 4 * g4 + j;
        float p = fast_exp2(__builtin_fmaf(sacc[reg], scale_log2, -l4[j]));
        if (decltype(masked)::value && my_key > qu + 8 * g4 + 4 * hf + j + shift) p = 0.f;
        pfr[reg >> 3][reg & 7] = f2bf(p);
        dsfr[reg >> 3][reg & 7] = f2bf(p * (pacc[reg] - d4[j]));
      }
    }
    // ---- dV^T += dO^T.P ; dK^T += Q^T.dS   (A operand from transposed reads, again a group ahead, the first ahead of the
    // exponentials: 24576 tokens 5590 -> 5546 us, 16384 6690 -> 6580)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int s = i >> 2, db = i & 3;
      if (i < 7) read_t(i + 1);
      __builtin_amdgcn_sched_barrier(0);
      dvacc[db] = mfma32(cat4(d0[i & 1], d1[i & 1]), pfr[s], dvacc[db]);
      dkacc[db] = mfma32(cat4(q0[i & 1], q1[i & 1]), dsfr[s], dkacc[db]);
    }
  };
  if (nwork > 0)
    issue();
  else
    dma_arrive();  // (V is on its way)
  dma_pin(kf);
  for (int h = 0; h < nh; ++h) {
    int sl = 0;
    for (; sl < n_diag; ++sl) {
      advance();
      if (kw0 <= (first + sl) * 32 + 31 + shift) step(sl, std::true_type{});  // otherwise no row sees a key of this wave
    }
    for (; sl < nslice; ++sl) {
      advance();
      step(sl, std::false_type{});
    }
  }
  // ---- epilogue: dK^T / dV^T accumulators: lane (key col = r, hf), reg -> d row
  if (my_key < k_len) {
    if (parts > 1) {
      float* pk = part + (((size_t)2 * pt * total_k + k_beg + my_key) * Hkv + kvh) * D;
      float* pv = pk + (size_t)total_k * Hkv * D;
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          f32x4 wk, wv;
#pragma unroll
          for (int j = 0; j < 4; ++j) { wk[j] = dkacc[db][4 * g4 + j]; wv[j] = dvacc[db][4 * g4 + j]; }
          *reinterpret_cast<f32x4*>(pk + 32 * db + 8 * g4 + 4 * hf) = wk;
          *reinterpret_cast<f32x4*>(pv + 32 * db + 8 * g4 + 4 * hf) = wv;
        }
      return;
    }
    bf16_t* dkp = dk + (size_t)(k_beg + my_key) * dk_stride + (size_t)kvh * D;
    bf16_t* dvp = dv + (size_t)(k_beg + my_key) * dv_stride + (size_t)kvh * D;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        bf16x4 wk, wv;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          wk[j] = f2bf(dkacc[db][4 * g4 + j] * softmax_scale);
          wv[j] = f2bf(dvacc[db][4 * g4 + j]);
        }
        *reinterpret_cast<bf16x4*>(dkp + 32 * db + 8 * g4 + 4 * hf) = wk;
        *reinterpret_cast<bf16x4*>(dvp + 32 * db + 8 * g4 + 4 * hf) = wv;
      }
  }
}

// dK, dV (bf16, strided) of the keys of the sequences = sum over the parts; grid (key blocks of 8, sequences): with
// blocks of 64 keys 700 tokens kept 11 workgroups busy for 31 us (two key heads)
__global__ __launch_bounds__(256) void flash_bwd_sum_kernel(const float* __restrict__ part, bf16_t* __restrict__ dk,
                                                            bf16_t* __restrict__ dv, const int* __restrict__ cu_k, int Hkv,
                                                            int64_t total_k, int parts, int64_t dk_stride,
                                                            int64_t dv_stride, float softmax_scale) {
  constexpr int D = 128;
  const int k_beg = cu_k[blockIdx.y], k_len = cu_k[blockIdx.y + 1] - k_beg;
  const int row0 = blockIdx.x * 8, rows = min(8, k_len - row0);
  const size_t all = (size_t)total_k * Hkv * D;
  for (int i = threadIdx.x; i < rows * Hkv * (D / 8); i += 256) {
    const int ch = i % (D / 8), rest = i / (D / 8), h = rest % Hkv;
    const int64_t tok = k_beg + row0 + rest / Hkv;
    const size_t at = ((size_t)tok * Hkv + h) * D + ch * 8;
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      f32x4 x = {}, y = {};
#pragma unroll 4
      for (int p = 0; p < parts; ++p) {
        const f32x4* s = reinterpret_cast<const f32x4*>(part + (2 * p + w) * all + at);
        x += s[0];
        y += s[1];
      }
      const float f = w == 0 ? softmax_scale : 1.f;
      bf16x8 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) { o[j] = f2bf(x[j] * f); o[j + 4] = f2bf(y[j] * f); }
      st8((w == 0 ? dk + tok * dk_stride : dv + tok * dv_stride) + (size_t)h * D + ch * 8, o);
    }
  }
}

// delta: [2, Hq, total_q] fp32 scratch (head size 256: [Hq, total_q] of it). part: [parts, 2, total_k, Hkv, D] fp32 scratch
// when parts > 1 (head size 128).
extern "C" int areal_flash_bwd(const void* q, const void* k, const void* v, const void* o,
                               const void* d_o, const float* lse, float* delta,
                               void* dq, void* dk, void* dv, float* part, int parts, const int* cu_q,
                               const int* cu_k, int B, int max_q, int max_k, int total_q, int64_t total_k, int Hq, int Hkv,
                               int D, int64_t q_stride, int64_t k_stride, int64_t v_stride,
                               int64_t o_stride, int64_t do_stride, int64_t dq_stride,
                               int64_t dk_stride, int64_t dv_stride, float softmax_scale, int causal,
                               hipStream_t st) {
  if (total_q == 0) return 0;
  if (D != 128 && D != 256) return -1;
  if (Hq % Hkv != 0) return -2;
  if ((q_stride | k_stride | v_stride | o_stride | do_stride | dq_stride | dk_stride | dv_stride) % 8)
    return -3;
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)d_o) % 16 != 0) return -4;
  if (q_stride > FLASH_MAX_STRIDE || k_stride > FLASH_MAX_STRIDE || v_stride > FLASH_MAX_STRIDE || do_stride > FLASH_MAX_STRIDE) return -5;
  if (D == 256)
    return areal_flash_bwd_d256(q, k, v, o, d_o, lse, delta, dq, dk, dv, cu_q, cu_k, B, max_k, total_q, total_k, Hq, Hkv,
                                q_stride, k_stride, v_stride, o_stride, do_stride, dq_stride, dk_stride, dv_stride,
                                softmax_scale, causal, st);
  {
    const FlashGrads grads{(bf16_t*)dq, (bf16_t*)dk, (bf16_t*)dv, dq_stride, dk_stride, dv_stride, total_q, total_k, cu_q, cu_k, B, Hkv};
    const int64_t n = (total_q > total_k ? total_q : total_k) * Hq * 16;
    hipLaunchKernelGGL(flash_bwd_delta_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                       (const bf16_t*)o, (const bf16_t*)d_o, lse, delta, o_stride, do_stride, Hq, total_q, grads);
  }
  const int G = Hq / Hkv, hs = (G + parts - 1) / parts;
  if (parts < 1 || parts > G || (parts > 1 && part == nullptr)) return -6;
  if (B == 0 || max_q == 0 || max_k == 0) return (int)hipGetLastError();  // no sequences, or none with rows
  const unsigned kblocks = (unsigned)((max_k + 127) / 128);
  hipLaunchKernelGGL(flash_bwd_dkv_kernel, dim3(kblocks * Hkv * B * parts), dim3(256), 0, st, (const bf16_t*)q,
                     (const bf16_t*)k, (const bf16_t*)v, (const bf16_t*)d_o, delta, (bf16_t*)dk, (bf16_t*)dv, part, cu_q,
                     cu_k, q_stride, k_stride, v_stride, do_stride, dk_stride, dv_stride, Hq, Hkv, B, total_q, total_k,
                     parts, hs, softmax_scale, causal);
  if (parts > 1)
    hipLaunchKernelGGL(flash_bwd_sum_kernel, dim3((max_k + 7) / 8, B), dim3(256), 0, st, part, (bf16_t*)dk, (bf16_t*)dv, cu_k,
                       Hkv, total_k, parts, dk_stride, dv_stride, softmax_scale);
  const int n_g_pad = (Hkv * B + 7) & ~7;
  dim3 qgrid((unsigned)(((max_q + 127) / 128) * (Hq / Hkv) * n_g_pad));
  hipLaunchKernelGGL(flash_bwd_dq_kernel, qgrid, dim3(256), 0, st, (const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v,
                     (const bf16_t*)d_o, delta, (bf16_t*)dq, cu_q, cu_k, q_stride, k_stride, v_stride, do_stride,
                     dq_stride, Hq, Hkv, B, total_q, softmax_scale, causal);
  return (int)hipGetLastError();
}
