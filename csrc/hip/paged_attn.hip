// Paged-KV decode attention, fused RoPE + KV-cache write and cache gather for gfx950.
//
// This is the rollout engine's replacement for flash_attn_with_kvcache
// (realhf/impl/model/modules/attn.py:272) and for the SGLang/vLLM paged attention the
// reference delegates to. The cache layout is chosen for the MFMA operand maps so the
// decode kernel needs no LDS staging and no transposes:
//
//   K cache  [num_pages, Hkv, 32, D]   (key-major rows of D)
//   V cache  [num_pages, Hkv, D, 32]   (stored TRANSPOSED: for one d, 32 keys contiguous)
//
// A page holds 32 tokens. For one page and one kv head:
//   S^T[key, q]  = K[key, :] . Q[q, :]        A = K rows (16 B per lane straight from HBM)
//   O^T[d, q]   += V^T[d, key] * P^T[key, q]  A = V^T rows (16 B per lane straight from HBM)
// with v_mfma_f32_16x16x32_bf16. The 16 "q" columns are the query heads that share the kv
// head (GQA group, zero padded). The two 16-key S^T tiles of a page take the keys
// {8c+r} and {8c+4+r} (c = lane>>4, r = 0..3) so that each lane ends up holding P for keys
// 8c..8c+7, which is exactly the B-operand order of the P.V product.
#include <type_traits>

#include "common.hpp"

#define PAGE 32

DEVINL f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// grid: (B, Hkv, nsplit); block: 256 threads = 4 waves. D = 64, 128 or 256 (template; 256 holds a page's 32 KiB of
// K and V fragments in registers and runs one workgroup per SIMD set instead of two).
// q: [B, Hq, D]; out: [B, Hq, D] when nsplit == 1 else partials.
// part_o: [B, Hq, nsplit, D] fp32, part_ml: [B, Hq, nsplit, 2] (m in log2 units, l).
// FP8: the caches hold e4m3 bytes (same layouts); a lane fetches 8 bytes per fragment and widens them to bf16 in
// registers - half the HBM traffic of the kernel, which is what bounds it at long contexts.
// WIN = true: the query (the context's last token) sees key j when ctx - 1 - j < window or j < keep (window <= 0:
// every key; chunk > 0: and floor(j / chunk) = floor((ctx - 1) / chunk)); pages without a visible key are skipped, and the softmax weights enter the P.V product as the pair
// (bf16(p), bf16(p - bf16(p))) so that they carry 16 bits of mantissa.
template <int D, bool FP8, bool WIN = false>
__global__ __launch_bounds__(256, (D > 128 ? 1 : 2)) void paged_decode_kernel(
    const bf16_t* __restrict__ q, const void* __restrict__ kcache,
    const void* __restrict__ vcache, const int* __restrict__ block_tables,
    const int* __restrict__ context_lens, bf16_t* __restrict__ out, float* __restrict__ part_o,
    float* __restrict__ part_ml, int Hq, int Hkv, int max_pages, float scale_log2, int q_stride, int window = 0,
    int keep = 0, const bf16_t* __restrict__ r1 = nullptr, const bf16_t* __restrict__ r2 = nullptr,
    const bf16_t* __restrict__ gate = nullptr, int64_t gate_stride = 0, int chunk = 0) {
  constexpr int KS = D / 32;  // k-steps of the QK product
  constexpr int DB = D / 16;  // 16-wide d blocks of the PV product
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int b = blockIdx.x, h = blockIdx.y, split = blockIdx.z, nsplit = gridDim.z;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int G = Hq / Hkv;
  const int col = lane & 15, c = lane >> 4;
  const int ctx = context_lens[b];
  const int npages = (ctx + PAGE - 1) / PAGE;
  // WIN: pages [0, n_keep) and [p_lo, npages) are walked; step i of the walk is page i (i < n_keep) or p_lo + i - n_keep
  const bool windowed = WIN && (window > 0 || chunk > 0);
  int first = windowed && window > 0 ? max(0, ctx - window) : 0;  // first key seen besides the kept ones
  if (windowed && chunk > 0) first = max(first, (ctx - 1) / chunk * chunk);
  const int p_lo = first / PAGE;
  const int n_keep = windowed ? min((max(keep, 0) + PAGE - 1) / PAGE, p_lo) : 0;
  const int nwalk = n_keep + npages - p_lo;
  const int per = (nwalk + nsplit - 1) / nsplit;
  const int p_beg = split * per;
  const int p_end = min(nwalk, p_beg + per);

  // Q as the B operand of S^T = K.Q^T: lane (q = col, c) holds Q[q][32ks + 8c + j]
  bf16x8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    if (col < G) qf[ks] = ld8(q + (size_t)b * q_stride + (size_t)(h * G + col) * D + ks * 32 + c * 8);
    else
#pragma unroll
      for (int j = 0; j < 8; ++j) qf[ks][j] = (bf16_t)0.f;
  }
  f32x4 o[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i) o[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;  // running max (log2 units) is shared by the 4 lanes of a q
  // WIN with r1 / r2: r1_h log2(1 + r2_h (ctx - 1 - j)) is taken off the score of this lane's query head
  const bool biased = WIN && r1 != nullptr && col < G;
  const float b1 = biased ? bf2f(r1[h * G + col]) : 0.f, b2 = biased ? bf2f(r2[h * G + col]) : 0.f;

  const int* bt = block_tables + (size_t)b * max_pages;
  for (int pi = p_beg + wid; pi < p_end; pi += 4) {
    const int p = pi < n_keep ? pi : p_lo + pi - n_keep;
    const int page = bt[p];
    const size_t kp = ((size_t)page * Hkv + h) * PAGE * D;  // element offsets of this page's K / V block
    const size_t vp = ((size_t)page * Hkv + h) * D * PAGE;
    // issue all loads of the page up front (16 KiB per wave in flight)
    bf16x8 ka[KS], kb[KS], vt[DB];
    const int key_a = 8 * (col >> 2) + (col & 3);  // row `col` of tile a
    const int key_b = key_a + 4;                   // row `col` of tile b
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      ka[ks] = ld8_cache<FP8>(kcache, kp + key_a * D + ks * 32 + c * 8);
      kb[ks] = ld8_cache<FP8>(kcache, kp + key_b * D + ks * 32 + c * 8);
    }
#pragma unroll
    for (int i = 0; i < DB; ++i) vt[i] = ld8_cache<FP8>(vcache, vp + (i * 16 + col) * PAGE + c * 8);

    f32x4 sa = {0.f, 0.f, 0.f, 0.f}, sb = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      sa = mfma16(ka[ks], qf[ks], sa);
      sb = mfma16(kb[ks], qf[ks], sb);
    }
    // lane (q = col, c): sa[r] = S[key 8c + r], sb[r] = S[key 8c + 4 + r]
    float s[8];
    const int key0 = p * PAGE + 8 * c;
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      float v = (r < 4 ? sa[r] : sb[r - 4]) * scale_log2;
      if (WIN && r1 != nullptr) v -= b1 * __log2f(1.f + b2 * (float)max(ctx - 1 - (key0 + r), 0));
      s[r] = (key0 + r < ctx && (!windowed || key0 + r >= first || key0 + r < keep)) ? v : -INFINITY;
      mx = fmaxf(mx, s[r]);
    }
    mx = max_xor16(mx);
    mx = max_xor32(mx);
    const float mn = fmaxf(m, mx);
    if (__any(mn > m)) {
      const float alpha = (m == -INFINITY) ? 0.f : fast_exp2(m - mn);
      l *= alpha;
#pragma unroll
      for (int i = 0; i < DB; ++i) o[i] *= alpha;
      m = mn;
    }
    bf16x8 pf, pl;
    float ls = 0.f;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const float pr = (m == -INFINITY) ? 0.f : fast_exp2(s[r] - m);
      ls += pr;
      pf[r] = f2bf(pr);
      if (WIN) pl[r] = f2bf(pr - bf2f(pf[r]));
    }
    l += ls;
    // O^T[d, q] += V^T[d, keys] . P^T[keys, q]
#pragma unroll
    for (int i = 0; i < DB; ++i) {
      o[i] = mfma16(vt[i], pf, o[i]);
      if (WIN) o[i] = mfma16(vt[i], pl, o[i]);
    }
  }
  // l is a per-lane partial over this lane's keys: sum the 4 lanes that share a q
  l = sum_xor16(l);
  l = sum_xor32(l);

  // combine the 4 waves through LDS: per wave [16 q][D] fp32 O + [16] m + [16] l
  // Rows are DP = D + 4 floats apart: with a stride of D floats the 16 q rows of a store fall on the same banks
  // (a 16-way conflict); 4 floats of padding move each row by one 16-byte slot, and each lane stores its 4
  // consecutive values as one 16-byte write. Only the G real q rows are stored.
  constexpr int DP = D + 4;
  float* so = smem;                 // [4][16][DP]
  float* sm = smem + 4 * 16 * DP;   // [4][16]
  float* sl = sm + 4 * 16;          // [4][16]
  if (col < G) {
#pragma unroll
    for (int i = 0; i < DB; ++i) *reinterpret_cast<f32x4*>(so + (wid * 16 + col) * DP + i * 16 + 4 * c) = o[i];
  }
  if (c == 0) { sm[wid * 16 + col] = m; sl[wid * 16 + col] = l; }
  __syncthreads();
  // thread t handles (q = t / (D/8)... ) : 256 threads cover G*D elements in a strided loop
  for (int idx = threadIdx.x; idx < G * D; idx += 256) {
    const int qq = idx / D, d = idx % D;
    float mm = -INFINITY;
#pragma unroll
    for (int w = 0; w < 4; ++w) mm = fmaxf(mm, sm[w * 16 + qq]);
    float acc = 0.f, ll = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float mw = sm[w * 16 + qq];
      const float f = (mw == -INFINITY) ? 0.f : fast_exp2(mw - mm);
      acc += so[(w * 16 + qq) * DP + d] * f;
      ll += sl[w * 16 + qq] * f;
    }
    const int head = h * G + qq;
    if (nsplit == 1) {
      float val = ll > 0.f ? acc / ll : 0.f;
      // WIN with a gate: one sigmoid gate per head and value channel of the row
      if (WIN && gate) val /= 1.f + __expf(-bf2f(gate[(size_t)b * gate_stride + (size_t)head * D + d]));
      out[(size_t)b * Hq * D + (size_t)head * D + d] = f2bf(val);
    } else {
      part_o[(((size_t)b * Hq + head) * nsplit + split) * D + d] = acc;
      if (d == 0) {
        part_ml[(((size_t)b * Hq + head) * nsplit + split) * 2 + 0] = mm;
        part_ml[(((size_t)b * Hq + head) * nsplit + split) * 2 + 1] = ll;
      }
    }
  }
}

// Combine split partials: grid (B * Hq), block D threads. The (max, sum) pairs of the splits are fetched by one
// parallel load into LDS and the partial outputs four splits at a time: a loop of one dependent load per split is a
// chain of memory round trips (16 splits at a batch of 8 rows: 7.5 us for a few KB).
__global__ void paged_decode_reduce_kernel(const float* __restrict__ part_o,
                                           const float* __restrict__ part_ml,
                                           bf16_t* __restrict__ out, int nsplit, int D,
                                           const bf16_t* __restrict__ gate = nullptr, int64_t gate_stride = 0,
                                           int Hq = 1) {
  constexpr int MAXS = 256;
  __shared__ float sm[MAXS], sl[MAXS];
  const int bh = blockIdx.x, d = threadIdx.x;
  const bool staged = nsplit <= MAXS;
  if (staged) {
    for (int s = d; s < nsplit; s += blockDim.x) {
      const float2 ml = *reinterpret_cast<const float2*>(part_ml + ((size_t)bh * nsplit + s) * 2);
      sm[s] = ml.x;
      sl[s] = ml.y;
    }
    __syncthreads();
  }
  auto M = [&](int s) { return staged ? sm[s] : part_ml[((size_t)bh * nsplit + s) * 2]; };
  auto Lsum = [&](int s) { return staged ? sl[s] : part_ml[((size_t)bh * nsplit + s) * 2 + 1]; };
  float mm = -INFINITY;
  for (int s = 0; s < nsplit; ++s) mm = fmaxf(mm, M(s));
  float acc = 0.f, ll = 0.f;
  const float* po = part_o + (size_t)bh * nsplit * D + d;
  int s = 0;
  for (; s + 4 <= nsplit; s += 4) {
    const float o0 = po[(size_t)s * D], o1 = po[(size_t)(s + 1) * D];
    const float o2 = po[(size_t)(s + 2) * D], o3 = po[(size_t)(s + 3) * D];
    const float os[4] = {o0, o1, o2, o3};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float ms = M(s + j);
      const float f = (ms == -INFINITY) ? 0.f : fast_exp2(ms - mm);
      acc += os[j] * f;
      ll += Lsum(s + j) * f;
    }
  }
  for (; s < nsplit; ++s) {
    const float ms = M(s);
    const float f = (ms == -INFINITY) ? 0.f : fast_exp2(ms - mm);
    acc += po[(size_t)s * D] * f;
    ll += Lsum(s) * f;
  }
  float val = ll > 0.f ? acc / ll : 0.f;
  if (gate) val /= 1.f + __expf(-bf2f(gate[(size_t)(bh / Hq) * gate_stride + (size_t)(bh % Hq) * D + d]));
  out[(size_t)bh * D + d] = f2bf(val);
}

template <int D, bool FP8>
static int launch_paged_decode(const void* q, const void* kcache, const void* vcache, const int* block_tables,
                               const int* context_lens, void* out, float* part_o, float* part_ml, int B, int Hq, int Hkv,
                               int max_pages, int nsplit, float scale_log2, int q_stride, hipStream_t st) {
  const size_t lds = (size_t)(4 * 16 * (D + 4) + 2 * 4 * 16) * sizeof(float);
  if (D == 256) {
    static bool attr_set = false;  // 67 KiB of dynamic LDS: above the default limit
    if (!attr_set) {
      HIP_RET(hipFuncSetAttribute((const void*)paged_decode_kernel<D, FP8>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)lds));
      attr_set = true;
    }
  }
  hipLaunchKernelGGL((paged_decode_kernel<D, FP8>), dim3(B, Hkv, nsplit), dim3(256), lds, st, (const bf16_t*)q, kcache,
                     vcache, block_tables, context_lens, (bf16_t*)out, part_o, part_ml, Hq, Hkv, max_pages, scale_log2,
                     q_stride);
  return 0;
}

// fp8: the caches hold e4m3 bytes instead of bf16 values
extern "C" int areal_paged_decode(const void* q, const void* kcache, const void* vcache,
                                  const int* block_tables, const int* context_lens, void* out,
                                  float* part_o, float* part_ml, int B, int Hq, int Hkv, int D,
                                  int max_pages, int nsplit, float softmax_scale, int q_stride, int fp8,
                                  hipStream_t st) {
  if (B == 0) return 0;
  if (Hq % Hkv != 0 || Hq / Hkv > 16) return -1;
  if (D != 128 && D != 64 && D != 256) return -2;
  if (nsplit < 1 || (nsplit > 1 && (!part_o || !part_ml))) return -3;
  const float scale_log2 = softmax_scale * 1.4426950408889634f;
  int rc = 0;
#define PD(DD, F8)                                                                                                    \
  rc = launch_paged_decode<DD, F8>(q, kcache, vcache, block_tables, context_lens, out, part_o, part_ml, B, Hq, Hkv,   \
                                   max_pages, nsplit, scale_log2, q_stride, st)
  if (D == 256) { if (fp8) PD(256, true); else PD(256, false); }
  else if (D == 128) { if (fp8) PD(128, true); else PD(128, false); }
  else { if (fp8) PD(64, true); else PD(64, false); }
#undef PD
  if (rc) return rc;
  if (nsplit > 1)
    hipLaunchKernelGGL(paged_decode_reduce_kernel, dim3(B * Hq), dim3(D), 0, st, part_o, part_ml,
                       (bf16_t*)out, nsplit, D);
  return (int)hipGetLastError();
}

// Decode over a sliding window that keeps the first `keep` tokens; bf16 caches, head sizes 64 / 128. r1 / r2 (one number
// per query head each, or null): a logarithmic distance penalty r1_h ln(1 + r2_h (i - j)) on the scaled scores. gate
// (rows of Hq D numbers, gate_stride apart, or null): the output is multiplied by sigmoid(gate) element by element.
extern "C" int areal_paged_decode_window(const void* q, const void* kcache, const void* vcache, const int* block_tables,
                                         const int* context_lens, void* out, float* part_o, float* part_ml, int B,
                                         int Hq, int Hkv, int D, int max_pages, int nsplit, float softmax_scale,
                                         int q_stride, int window, int keep, const void* r1, const void* r2,
                                         const void* gate, int64_t gate_stride, int chunk, hipStream_t st) {
  if (B == 0) return 0;
  if (Hq % Hkv != 0 || Hq / Hkv > 16) return -1;
  if (D != 128 && D != 64) return -2;
  if (nsplit < 1 || (nsplit > 1 && (!part_o || !part_ml))) return -3;
  const float scale_log2 = softmax_scale * 1.4426950408889634f;
  const size_t lds = (size_t)(4 * 16 * (D + 4) + 2 * 4 * 16) * sizeof(float);
  if (D == 128)
    hipLaunchKernelGGL((paged_decode_kernel<128, false, true>), dim3(B, Hkv, nsplit), dim3(256), lds, st,
                       (const bf16_t*)q, kcache, vcache, block_tables, context_lens, (bf16_t*)out, part_o, part_ml, Hq,
                       Hkv, max_pages, scale_log2, q_stride, window, keep, (const bf16_t*)r1, (const bf16_t*)r2,
                       (const bf16_t*)gate, gate_stride, chunk);
  else
    hipLaunchKernelGGL((paged_decode_kernel<64, false, true>), dim3(B, Hkv, nsplit), dim3(256), lds, st,
                       (const bf16_t*)q, kcache, vcache, block_tables, context_lens, (bf16_t*)out, part_o, part_ml, Hq,
                       Hkv, max_pages, scale_log2, q_stride, window, keep, (const bf16_t*)r1, (const bf16_t*)r2,
                       (const bf16_t*)gate, gate_stride, chunk);
  if (nsplit > 1)
    hipLaunchKernelGGL(paged_decode_reduce_kernel, dim3(B * Hq), dim3(D), 0, st, part_o, part_ml, (bf16_t*)out, nsplit, D,
                       (const bf16_t*)gate, gate_stride, Hq);
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------
// The same attention on a list of work items of near-equal size (one row and a range of its pages each), so that rows
// of very different length load the chip evenly, and without a second launch for the combination.
//
// What bounds it: HBM streaming of the pages. Measured per layer (12 query heads on 2 key heads of 128 unless said), one
// split count for all rows and a second launch -> items of about 1/256 of the batch and workgroups of 8 waves, two a CU:
//   1 x 640 10.0 -> 7.0 us (latency), 24 x 200-4096 22.4 -> 15.4, 320 x 128-1152 53.6 -> 42.4 (3.9 -> 4.9 TB/s),
//   256 x 640 32.3 -> 32.7 (even already), 64 x 128-1152 with 32 on 4 heads 25.8 -> 24.8, 1 x 16000 16.2 -> 16.3,
//   fp8: 48 x 6000-24000 101 -> 77 (3.6 -> 4.7 TB/s), 24 x 200-4096 17.7 -> 11.0, 128 x 1000 21.4 -> 16.1.
// More, smaller items cost more in combining than they even out (24 x 200-4096: 15.4 us with 256 items, 18.2 with 384;
// 320 x 128-1152, every row divided by its length over the item's rounded up: 42 with 256, 46 with 768-1024).
// The list depends on the context lengths alone (`stream` on the block tables): one launch per decode step serves every layer.
//
// Item: {row, first page, end page, first partial result of the row, number of the row's items, this item's partial
// result, whether its pages are read past the caches} in 8 ints; count 0: none. Longest first: a workgroup that ends early takes the
// next item, and the short ones fill the gaps at the end.
struct DecodeItem { int b, p_beg, p_end, base, n, part, stream, pad; };

// Pages per item of a row of np pages: the row evenly divided into items of about `even` pages (half as much again at
// most: splitting a row that is a little longer than an item costs more than it evens out), a multiple of STEP; and so
// many that the workgroup that combines a row's n partial results does not read longer than the others walk:
// n^2 <= 3 pages (1 x 16000 tokens: 16.3 us, 22.4 us with n^2 <= 5 pages of 4-page items).
constexpr int STEP = 4;
// The number of items doubles (paged_decode_items_kernel) where one of them would be 1.4 times the even share, or where there
// are more of them than CUs for a key head (`target`) but not twice as many: then some CUs get two items of a whole share each
// and the others one. Shares below 32, respectively 40 pages never double: the combination costs more than it evens out.
// Over 335 batches (1 to 384 rows, equal and ragged lengths to 24000, bf16 and fp8, 1 to 8 key heads of 64 and 128) the layout
// that this picks takes 0.5 % more than the better one, at most 14 %; the first condition alone 2.1 % and 36 %. us a layer,
// one split count for all rows / items / items doubled, 12 query heads on 2: 48 equal rows of 6000 tokens 62 / 73 / 58 (144 items
// on 128 CUs), 80 of 6000 106 / 109 / 91, 60 of 3000-9000 87 / 103 / 73, 90 of 2000-7000 116 / 112 / 84; not doubled: 100 of
// 6000 111 / 105 / 122 (1.28 times the share), 16 of 12000 41 / 40 / 43, 8 of 4000-16000 23 / 20 / 23 (shares of 16).
constexpr int FINER_EVEN = 32, FINER_COUNT_EVEN = 40;
constexpr int MAX_ROW_ITEMS = 256;  // (reached at 699000 tokens) their (m, l) fit the LDS that the waves' results need, 8 (64 + 4) floats a head
DEVINL int pages_per_item(int np, int even) {
  const int most = min(MAX_ROW_ITEMS, max(1, (int)sqrtf(3.f * (float)np)));
  const int n = min(most, max(1, (np + even / 2) / even));
  const int per = (np + n - 1) / n;
  return max(STEP, (per + STEP - 1) / STEP * STEP);
}

// grid 1, block 1024. n_items >= min(target + B, the rows' largest number of items x B),
// with `finer` 2 target + B. Pages per item: the whole batch over `target` items.
__global__ __launch_bounds__(1024) void paged_decode_items_kernel(const int* __restrict__ context_lens,
                                                                  DecodeItem* __restrict__ items, int2* __restrict__ rows,
                                                                  int B, int target, int n_items, int finer,
                                                                  const int* __restrict__ block_tables, int max_pages) {
  constexpr int NB = 64;  // size classes of the sort
  // For the items' `stream`, page ids in an open-addressed table. First the rows' first pages: batches in which no row shares its own are done
  // with that. Where some do (requests of one prompt, several prompts behind one system prompt), the middle pages of their items, and what
  // such rows have in these places is looked up and counted: 320 rows with 1024 tokens common to 16 each 6.4 -> 8.8 us, 1024 rows 8.9 -> 12.5,
  // none shared 6.4. (Compared with one row of the same first page only, the pages of several prompts behind a system prompt went past the
  // caches: 320 x 1100-1152, 64 tokens common to all and 960 to 16 each, 53.3 us a layer, now 40.7; 64 x 4150, 256 and 3840 to 8, 38.7 and
  // 29.4.) 1024 rows at most; a page that finds no place in PROBES counts as shared. A row of one page (a bucket's idle rows among them)
  // writes into it and has it to itself.
  constexpr int SLOTS = 4096, PROBES = 32;
  __shared__ __attribute__((aligned(16))) int key[SLOTS], seen[SLOTS];
  __shared__ int mate_pages[1024];
  constexpr int PLACES = 8192, NI = 2;  // of a row's pages, and items a thread; what lies further on counts as shared
  __shared__ unsigned listed[PLACES / 32];
  __shared__ unsigned short place[NI * 1024];
  __shared__ int places;
  const bool shared_pages = block_tables && B > 1 && B <= 1024;
  __shared__ int red[16], red_n[16], hist[NB];
  const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
  auto slot_of = [&](int page) __attribute__((always_inline)) { return (unsigned)page * 2654435761u >> 20; };
  auto find = [&](int page, bool put) __attribute__((always_inline)) {  // the page's slot, or -1
    unsigned at = slot_of(page);
    for (int i = 0; i < PROBES; ++i, at = (at + 1) & (SLOTS - 1)) {
      const int had = put ? atomicCAS(&key[at], -1, page) : key[at];
      if (had == page || (put && had == -1)) return (int)at;
      if (had == -1) break;
    }
    return -1;
  };
  auto clear = [&]() __attribute__((always_inline)) {
    static_assert(SLOTS == 4 * 1024);
    *reinterpret_cast<int4*>(&key[4 * t]) = make_int4(-1, -1, -1, -1);
    *reinterpret_cast<int4*>(&seen[4 * t]) = make_int4(0, 0, 0, 0);
  };
  int own_first = 0, own_slot = -1, own_pages = 0;
  if (shared_pages) {
    own_first = block_tables[(size_t)min(t, B - 1) * max_pages];
    own_pages = t < B ? min((max(context_lens[t], 0) + PAGE - 1) / PAGE, max_pages) : 0;
    clear();
  }
  int pages = 0;
  for (int b = t; b < B; b += 1024) pages += (max(context_lens[b], 0) + PAGE - 1) / PAGE;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) pages += __shfl_xor(pages, o, 64);
  if (lane == 0) red[wid] = pages;
  if (t < NB) hist[t] = 0;
  __syncthreads();
  int total = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) total += red[w];
  if (own_pages > 1) {
    own_slot = find(own_first, true);
    if (own_slot >= 0) atomicAdd(&seen[own_slot], 1);
  }
  int even = max(STEP, (total + target - 1) / target);
  if (finer && even >= FINER_EVEN) {
    int longest = 0, count = 0;
    for (int b = t; b < B; b += 1024) {
      const int np = (max(context_lens[b], 0) + PAGE - 1) / PAGE, per = pages_per_item(np, even);
      longest = max(longest, per);
      count += max(1, (np + per - 1) / per);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      longest = max(longest, __shfl_xor(longest, o, 64));
      count += __shfl_xor(count, o, 64);
    }
    __syncthreads();
    if (lane == 0) { red[wid] = longest; red_n[wid] = count; }
    __syncthreads();
    count = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      longest = max(longest, red[w]);
      count += red_n[w];
    }
    if (5 * longest > 7 * even || (even >= FINER_COUNT_EVEN && count > target && count <= 2 * target))
      even = max(STEP, (total + 2 * target - 1) / (2 * target));
    __syncthreads();
  }
  const int top = even + even / 2 + STEP;  // an item has more pages only if its row may not be divided further
  auto size_class = [&](int size) { return NB - 1 - min(NB - 1, size * (NB - 1) / top); };
  for (int b = t; b < B; b += 1024) {  // items per size class
    const int np = (max(context_lens[b], 0) + PAGE - 1) / PAGE, per = pages_per_item(np, even);
    const int n = max(1, (np + per - 1) / per);
    if (n > 1) atomicAdd(&hist[size_class(per)], n - 1);
    atomicAdd(&hist[size_class(np - (n - 1) * per)], 1);
  }
  __syncthreads();
  if (t < NB) {  // first place of every class (64 lanes: one wave)
    int incl = hist[t];
    const int own = incl;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o, 64);
      if (lane >= o) incl += v;
    }
    hist[t] = incl - own;
  }
  int at = 0;  // items of the rows before this pass over 1024 rows
  for (int b0 = 0; b0 < B; b0 += 1024) {
    const int b = b0 + t;
    const int np = b < B ? (max(context_lens[b], 0) + PAGE - 1) / PAGE : 0;
    const int per = pages_per_item(np, even);
    const int n = b < B ? max(1, (np + per - 1) / per) : 0;
    int incl = n;  // prefix sum over the block
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o, 64);
      if (lane >= o) incl += v;
    }
    __syncthreads();
    if (lane == 63) red[wid] = incl;
    __syncthreads();
    int before = at;
    for (int w = 0; w < 16; ++w) {
      if (w < wid) before += red[w];
      at += red[w];
    }
    const int base = before + incl - n;
    if (n > 0 && rows) rows[b] = base + n <= n_items ? make_int2(base, n) : make_int2(0, 0);
    for (int i = 0; i < n; ++i) {
      const int lo = i * per, hi = min(np, lo + per), stream = B == 1 || shared_pages;
      const int place = atomicAdd(&hist[size_class(hi - lo)], 1);
      if (place < n_items && base + n <= n_items) items[place] = DecodeItem{b, lo, hi, base, n, base + i, stream, 0};
    }
  }
  for (int i = at + t; i < n_items; i += 1024) items[i] = DecodeItem{0, 0, 0, 0, 0, 0, 0, 0};

  if (!shared_pages) return;
  // Pages that other rows read too. (A row's first slot was filled ahead of the barriers above.)
  const bool mate = own_pages > 1 && (own_slot < 0 || seen[own_slot] > 1);
  if (!__syncthreads_or(mate)) return;
  clear();
  mate_pages[t] = mate ? own_pages : 0;
  if (t < PLACES / 32) listed[t] = 0;
  if (t == 0) places = 0;
  __syncthreads();
  const int n_at = min(at, n_items);
  int slot[NI];
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const int i = t + 1024 * j;
    slot[j] = -2;  // no other row's
    if (i < n_at) {
      const DecodeItem it = items[i];
      const int mid = min((it.p_beg + it.p_end) / 2, max_pages - 1);
      if (mate_pages[it.b] > 0) {
        slot[j] = mid < PLACES ? find(block_tables[(size_t)it.b * max_pages + mid], true) : -1;
        if (mid < PLACES && !(atomicOr(&listed[mid >> 5], 1u << (mid & 31)) >> (mid & 31) & 1)) place[atomicAdd(&places, 1)] = mid;
      }
    }
  }
  __syncthreads();
  // A page that rows share is in the same place of each: the rows' pages in the places where some item has its middle.
  const int all = places * B;
  for (int i0 = t; i0 < all; i0 += 1024 * 4) {
    int page[4];
    bool have[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = i0 + 1024 * u, b = i / places, p = i < all ? place[i - b * places] : 0;
      have[u] = i < all && p < mate_pages[b];
      page[u] = have[u] ? block_tables[(size_t)b * max_pages + p] : 0;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int s = have[u] ? find(page[u], false) : -1;
      if (s >= 0) atomicAdd(&seen[s], 1);
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NI; ++j)
    if (slot[j] == -1 || (slot[j] >= 0 && seen[slot[j]] > 1)) items[t + 1024 * j].stream = 0;
  for (int i = t + 1024 * NI; i < n_at; i += 1024) items[i].stream = 0;
}

// Partial results travel between workgroups of any XCD: stores and loads at agent scope go past the XCD's own L2, so a
// store that has been waited for (vmcnt) is seen by every later load of this kind. Nothing else has to be written back or
// invalidated: acquire / release at agent scope on the counter would flush the whole L2 for each workgroup (measured:
// 93 instead of 34 us for 256 rows of 640 tokens in two items each).
DEVINL void st_agent(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
DEVINL float ld_agent(const float* p) {
  return __hip_atomic_load(const_cast<float*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// grid: n_items x Hkv, the heads of an item beside each other and the empty items last (workgroups that exit at once, spread
// among the others, leave some CUs with two and some with none: 120 instead of 96 us for 64 rows of 4000 tokens, 4 heads);
// block: NW waves, page by page in turn. part_o: [n_items, Hq, D], part_ml: [n_items, Hq, 2],
// arrived: [B, Hkv] zeros, zeros again afterwards. The last workgroup of a row to arrive combines its partial results
// in the order of the items: the result does not depend on the order of arrival.
// A wave is never without requests: the next page's K is asked for as soon as this page's scores have used up its registers, the
// next V behind the second product; Q, whose registers that takes, is read from LDS. us a layer, page after page -> this, 12 query
// heads on 2 of 128: 1 x 640 7.2 -> 6.9, 24 x 200-4096 16.0 -> 15.7, 256 x 640 32.1 -> 31.7, 320 x 128-1152 43.3 -> 43.2, 16 x 12000
// 40.8 -> 38.8, 384 x 8-64 8.2 -> 7.5, fp8 48 x 6000-24000 81.0 -> 81.8, 128 x 1000 15.3 -> 14.9; 14 on 2 of 64, 300 x 100-1200 23.8 ->
// 22.6; 8 on 1 of 256, 64 x 1000 22.1 -> 21.4, fp8 32 x 8000 34.9 -> 33.4, 1 x 640 12.5 -> 12.8: 4.8 to 5.6 of the 6 TB/s that the
// chip reads, less where a launch is over in 10 us.
// Pages are asked for in whole 128-byte lines, and where no other row reads them too, past the caches (nontemporal): lines alone gain nothing,
// the second alone 0 to 8 %, both 7 to 12: 320 x 128-1152 44.0 -> 39.6, 256 x 640 33.1 -> 29.9 (5.6 TB/s), 64 x 4000 52.0 -> 47.0, 24 x 200-4096
// 16.6 -> 15.3, 16 x 12000 40.9 -> 37.2, fp8 48 x 6000-24000 74.0 -> 67.0, 128 x 1000 15.7 -> 14.2; 300 x 100-1200 14 on 2 of 64 22.8 -> 20.4; 64 x 1000 8
// on 1 of 256 21.5 -> 20.2, fp8 32 x 8000 33.5 -> 30.7; 1 x 640 7.3 -> 7.0, 320 x 8-64 8.1. Pages of a common prompt come out of the caches for
// all rows but the first; past them, 320 x 1100-1152 with 1024 tokens common to 16 rows each took 51.4 instead of 44.0, 64 x 4150 with 4096
// common to 8 rows 40.6 instead of 31.2. The page loop is there twice; a wave's number is a scalar, so that both fit the registers. What
// stands ahead of the first request is on every launch's path: without a division and with the item read at once, 0.2 us less.
// LDS holds the G real query rows only. Two workgroups of 8 waves a CU (128 registers a lane; heads of 64 three, of 256 one
// of 4 waves): the register file sets that, a GQA group of 6 heads of 128 takes 26 KB of LDS.
template <int D, bool FP8, int NW>
__global__ __launch_bounds__(64 * NW, (D > 128 ? 1 : 4)) void paged_decode_walk_kernel(
    const bf16_t* __restrict__ q, const void* __restrict__ kcache, const void* __restrict__ vcache,
    const int* __restrict__ block_tables, const int* __restrict__ context_lens, const DecodeItem* __restrict__ items,
    bf16_t* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml, int* __restrict__ arrived, int Hq,
    int Hkv, int G, unsigned hkv_inv, int max_pages, float scale_log2, int q_stride) {
  constexpr int KS = D / 32, DB = D / 16, DP = D + 4;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  __shared__ int last;
  const int item = quotient(blockIdx.x, Hkv, hkv_inv);
  const DecodeItem it = items[item];
  // the whole item and the arguments at once, not each where it is first used: every wait is a trip to the scalar cache or past it
  int count = it.n;
  asm("" : "+s"(count) : "s"(it.b), "s"(it.p_beg), "s"(it.p_end), "s"(it.base), "s"(it.part), "s"(it.stream), "s"(q), "s"(kcache), "s"(vcache),
      "s"(block_tables), "s"(context_lens), "s"(G), "s"(q_stride));
  if (count == 0) return;
  const int b = it.b, h = blockIdx.x - item * Hkv;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, c = lane >> 4;
  const int* bt = block_tables + (size_t)b * max_pages;
  // this wave's pages: p_beg + wid + NW i; 64 page ids are fetched at once, one a lane
  const int mine = it.p_end - it.p_beg > wid ? (it.p_end - it.p_beg - wid + NW - 1) / NW : 0;
  int ids = 0;
  const int ctx = context_lens[b];
  // Q is the B operand of S^T = K.Q^T and waits in the LDS that the wave's result goes to at the end: its registers hold the next
  // page instead. fp8: a lane's 16 loaded bytes of K are the operand of two k-steps, so lane c takes Q[64 (ks / 2) + 16 c +
  // 8 (ks % 2) + j] there and Q[32 ks + 8 c + j] otherwise. Columns from G on repeat the last one and are not stored.
  constexpr int QP = D + 8;  // row pitch: 16-byte reads of 16 rows on different banks
  bf16_t* qs = reinterpret_cast<bf16_t*>(smem + wid * G * DP);
  if (mine > 0) {
    ids = bt[it.p_beg + wid + NW * min(lane, mine - 1)];
    const unsigned chunks = G * (D / 8);
    const bf16_t* qp = q + (size_t)b * q_stride + (size_t)h * G * D;
    bf16x8 qv[D / 32];
#pragma unroll
    for (int j = 0; j < D / 32; ++j) qv[j] = ld8(qp + min(lane + 64u * j, chunks - 1) * 8);
#pragma unroll
    for (int j = 0; j < D / 32; ++j) {
      const unsigned i = min(lane + 64u * j, chunks - 1);  // (the last piece more than once)
      st8(qs + i / (D / 8) * QP + i % (D / 8) * 8, qv[j]);
    }
  }
  const bf16_t* qrow = qs + min(col, G - 1) * QP + c * (FP8 ? 16 : 8);
  auto qf = [&](int ks) __attribute__((always_inline)) { return ld8(qrow + (FP8 ? (ks >> 1) * 64 + (ks & 1) * 8 : ks * 32)); };
  f32x4 o[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i) o[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;  // running max (log2 units) is shared by the 4 lanes of a q

  // Element offset of the K / V block of this wave's page i. The wait belongs to the fetch: behind the branch it would hold
  // every page's loads.
  auto block_of = [&](int i) __attribute__((always_inline)) {
    if (i > 0 && (i & 63) == 0) {
      ids = lane + i < mine ? bt[it.p_beg + wid + NW * (lane + i)] : 0;
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    }
    return ((size_t)__builtin_amdgcn_readlane(ids, i & 63) * Hkv + h) * PAGE * D;
  };
  // K and V of a page as loaded, 16 KiB (fp8: 8 KiB) a wave
  using kraw = std::conditional_t<FP8, u32x4, bf16x8>;
  using vraw = std::conditional_t<FP8, u32x2, bf16x8>;
  constexpr int KL = FP8 ? KS / 2 : KS;
  kraw ra[KL], rb[KL];
  vraw rv[DB];
  // a page's base is the same for all lanes, a lane's offset is the same for all pages: scalar base + 32-bit offset
  constexpr int EB = FP8 ? 1 : 2;
  // Row r of score tile a is key 8 (r / 4) + r % 4, of tile b the key 4 further. A request asks for whole 128-byte lines: of eight rows, lanes
  // with col >= 8 the second 64 bytes of what an operand would take of sixteen, and `sort` puts the halves of two requests in order.
  constexpr bool LINES = KL > 1;
  const int krow = LINES ? col & 7 : col;
  const unsigned k_off = (8 * (krow >> 2) + (krow & 3)) * D * EB + (LINES ? (col >> 3) * 64 : 0) + c * 16, v_off = (col * PAGE + c * 8) * EB;
  auto load_k = [&](size_t kp, auto stream_c) __attribute__((always_inline)) {
    constexpr bool STREAM = decltype(stream_c)::value;
    const char* base = reinterpret_cast<const char*>(kcache) + kp * EB;
#pragma unroll
    for (int k2 = 0; k2 < KL; ++k2) {
      const char* rows = base + (k2 & 1) * 16 * D * EB;  // rows 8 to 15 of the tiles
      const kraw* pa = reinterpret_cast<const kraw*>(rows + k_off + (k2 >> 1) * 128);
      const kraw* pb = reinterpret_cast<const kraw*>(rows + k_off + 4 * D * EB + (k2 >> 1) * 128);
      ra[k2] = STREAM ? __builtin_nontemporal_load(pa) : *pa;
      rb[k2] = STREAM ? __builtin_nontemporal_load(pb) : *pb;
    }
  };
  // a: the halves of rows 0 to 7 (lanes below and from col 8), b: of rows 8 to 15 -> the first halves of all rows, the second halves
  auto sort = [&](kraw& a, kraw& b) __attribute__((always_inline)) {
    u32x4 x = __builtin_bit_cast(u32x4, a), y = __builtin_bit_cast(u32x4, b);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      constexpr int ROTATE_8 = 0x128;  // within 16 lanes; the last arguments: of which groups of four lanes
      const unsigned first = __builtin_amdgcn_update_dpp(x[i], y[i], ROTATE_8, 0xF, 0xC, false);
      y[i] = __builtin_amdgcn_update_dpp(y[i], x[i], ROTATE_8, 0xF, 0x3, false);
      x[i] = first;
    }
    a = __builtin_bit_cast(kraw, x);
    b = __builtin_bit_cast(kraw, y);
  };
  auto load_v = [&](size_t kp, auto stream_c) __attribute__((always_inline)) {
    constexpr bool STREAM = decltype(stream_c)::value;
    const char* base = reinterpret_cast<const char*>(vcache) + kp * EB;
#pragma unroll
    for (int j = 0; j < DB; ++j) {
      const vraw* p = reinterpret_cast<const vraw*>(base + (j * 16 * PAGE * EB & ~4095) + v_off + (j * 16 * PAGE * EB & 4095));
      rv[j] = STREAM ? __builtin_nontemporal_load(p) : *p;
    }
  };
  auto page_step = [&](int p, size_t next, auto more_c, auto stream_c) __attribute__((always_inline)) {
    constexpr bool MORE = decltype(more_c)::value;  // another page follows
    f32x4 sa = {0.f, 0.f, 0.f, 0.f}, sb = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k2 = 0; k2 + 1 < KL; k2 += 2) {
      sort(ra[k2], ra[k2 + 1]);
      sort(rb[k2], rb[k2 + 1]);
    }
    if constexpr (FP8) {
#pragma unroll
      for (int k2 = 0; k2 < KL; ++k2) {
        sa = mfma16(fp8x8_to_bf16((u32x2){ra[k2][0], ra[k2][1]}), qf(2 * k2), sa);
        sb = mfma16(fp8x8_to_bf16((u32x2){rb[k2][0], rb[k2][1]}), qf(2 * k2), sb);
        sa = mfma16(fp8x8_to_bf16((u32x2){ra[k2][2], ra[k2][3]}), qf(2 * k2 + 1), sa);
        sb = mfma16(fp8x8_to_bf16((u32x2){rb[k2][2], rb[k2][3]}), qf(2 * k2 + 1), sb);
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        sa = mfma16(ra[ks], qf(ks), sa);
        sb = mfma16(rb[ks], qf(ks), sb);
      }
    }
    if (MORE) {
      __builtin_amdgcn_sched_barrier(0);
      load_k(next, stream_c);
      __builtin_amdgcn_sched_barrier(0);
    }
    // lane (q = col, c): sa[r] = S[key 8c + r], sb[r] = S[key 8c + 4 + r]
    float s[8];
    const int key0 = p * PAGE + 8 * c;
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const float v = (r < 4 ? sa[r] : sb[r - 4]) * scale_log2;
      s[r] = key0 + r < ctx ? v : -INFINITY;
      mx = fmaxf(mx, s[r]);
    }
    mx = max_xor16(mx);
    mx = max_xor32(mx);
    const float mn = fmaxf(m, mx);
    if (__any(mn > m)) {
      const float alpha = (m == -INFINITY) ? 0.f : fast_exp2(m - mn);
      l *= alpha;
#pragma unroll
      for (int j = 0; j < DB; ++j) o[j] *= alpha;
      m = mn;
    }
    bf16x8 pf;
    float ls = 0.f;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const float pr = (m == -INFINITY) ? 0.f : fast_exp2(s[r] - m);
      ls += pr;
      pf[r] = f2bf(pr);
    }
    l += ls;
    // O^T[d, q] += V^T[d, keys] . P^T[keys, q]
#pragma unroll
    for (int j = 0; j < DB; ++j) {
      if constexpr (FP8) o[j] = mfma16(fp8x8_to_bf16(rv[j]), pf, o[j]);
      else o[j] = mfma16(rv[j], pf, o[j]);
    }
    if (MORE) {
      __builtin_amdgcn_sched_barrier(0);
      load_v(next, stream_c);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto walk = [&](auto stream_c) __attribute__((always_inline)) {
    size_t kp = block_of(0);
    load_k(kp, stream_c);
    load_v(kp, stream_c);
    __builtin_amdgcn_sched_barrier(0);
    const int p0 = it.p_beg + wid;
    for (int i = 0; i + 1 < mine; ++i) {
      kp = block_of(i + 1);
      page_step(p0 + NW * i, kp, std::true_type{}, stream_c);
    }
    page_step(p0 + NW * (mine - 1), 0, std::false_type{}, stream_c);
  };
  if (mine > 0) {
    if (__builtin_expect(it.stream != 0, 1)) walk(std::true_type{});
    else walk(std::false_type{});
  }
  l = sum_xor16(l);  // l is a per-lane partial over this lane's keys: sum the 4 lanes that share a q
  l = sum_xor32(l);

  // combine the waves through LDS: rows DP floats apart keep the 16-byte stores of a wave's rows on different banks
  float* so = smem;                // [NW][G][DP]
  float* sm = smem + NW * G * DP;  // [NW][16]
  float* sl = sm + NW * 16;        // [NW][16]
  if (col < G) {
#pragma unroll
    for (int j = 0; j < DB; ++j) *reinterpret_cast<f32x4*>(so + (wid * G + col) * DP + j * 16 + 4 * c) = o[j];
  }
  if (c == 0) { sm[wid * 16 + col] = m; sl[wid * 16 + col] = l; }
  __syncthreads();
  for (int idx = threadIdx.x; idx < G * D; idx += 64 * NW) {
    const int qq = idx / D, d = idx % D;
    float mm = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) mm = fmaxf(mm, sm[w * 16 + qq]);
    float acc = 0.f, ll = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float mw = sm[w * 16 + qq];
      const float f = (mw == -INFINITY) ? 0.f : fast_exp2(mw - mm);
      acc += so[(w * G + qq) * DP + d] * f;
      ll += sl[w * 16 + qq] * f;
    }
    const int head = h * G + qq;
    if (it.n == 1) {
      out[((size_t)b * Hq + head) * D + d] = f2bf(ll > 0.f ? acc / ll : 0.f);
    } else {
      const size_t row = (size_t)it.part * Hq + head;
      st_agent(part_o + row * D + d, acc);
      if (d == 0) {
        st_agent(part_ml + row * 2, mm);
        st_agent(part_ml + row * 2 + 1, ll);
      }
    }
  }
  if (it.n == 1 || !arrived) return;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every wave's stores have arrived ...
  __syncthreads();
  if (threadIdx.x == 0) {                           // ... before the workgroup is counted
    const int old = __hip_atomic_fetch_add(arrived + (size_t)b * Hkv + h, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last = old == it.n - 1;
    if (last) __hip_atomic_store(arrived + (size_t)b * Hkv + h, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!last) return;
  // (m, l) of the row's items, [n][G][2], in the place of the waves' results; then U values a thread and eight items of
  // each in flight: ceil(n / 8) round trips past the L2. With one value at a time and its own (m, l) they were ceil(G D / threads)
  // times as many: 12 heads on 2, 2 rows of 24000 tokens 21.6 us a layer and 19.8 now, 8 of 8000 18.2 and 17.7; 32 on 4, 2 rows
  // of 1000-24000 20.8 and 18.9; 16 on one, 8 of 4000-16000 27.5 and 23.9.
  float* mls = smem;
  const size_t row0 = (size_t)it.base * Hq + h * G;
  for (int i = threadIdx.x; i < it.n * 2 * G; i += 64 * NW) mls[i] = ld_agent(part_ml + (row0 + (size_t)(i / (2 * G)) * Hq) * 2 + i % (2 * G));
  __syncthreads();
  auto combine = [&](auto u_c) {
    constexpr int U = decltype(u_c)::value;
    for (int i0 = threadIdx.x; i0 < G * D; i0 += U * 64 * NW) {
      float mm[U], acc[U], ll[U];
#pragma unroll
      for (int u = 0; u < U; ++u) { mm[u] = -INFINITY; acc[u] = 0.f; ll[u] = 0.f; }
      for (int s0 = 0; s0 < it.n; s0 += 8) {
        float os[U][8];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int j = 0; j < 8; ++j)
            os[u][j] = ld_agent(part_o + (row0 + (size_t)min(s0 + j, it.n - 1) * Hq) * D + min(i0 + u * 64 * NW, G * D - 1));
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const float* ml = mls + min(i0 + u * 64 * NW, G * D - 1) / D * 2;
          float ms[8], mn = mm[u];
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            ms[j] = s0 + j < it.n ? ml[(s0 + j) * 2 * G] : -INFINITY;
            mn = fmaxf(mn, ms[j]);
          }
          const float f0 = mm[u] == -INFINITY ? 0.f : fast_exp2(mm[u] - mn);
          acc[u] *= f0;
          ll[u] *= f0;
          mm[u] = mn;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float f = ms[j] == -INFINITY ? 0.f : fast_exp2(ms[j] - mn);
            acc[u] += os[u][j] * f;
            ll[u] += ml[min(s0 + j, it.n - 1) * 2 * G + 1] * f;
          }
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (i0 + u * 64 * NW < G * D)
          out[((size_t)b * Hq + h * G) * D + i0 + u * 64 * NW] = f2bf(ll[u] > 0.f ? acc[u] / ll[u] : 0.f);
    }
  };
  if constexpr (16 * D > 2 * 64 * NW) {
    if (G * D > 2 * 64 * NW) return combine(std::integral_constant<int, 4>{});
  }
  combine(std::integral_constant<int, 2>{});
}

// Items of the batch's decode attention; rows [B] (or null): first partial result and number of a row's items; `items`: n_items x 8 ints, at least min(target + B, B x most items of a row); with finer 2 target + B.
// block_tables [B, max_pages] (or null): pages that no other row reads are then read past the caches.
extern "C" int areal_paged_decode_items(const int* context_lens, void* items, void* rows, int B, int target, int n_items, int finer,
                                        const int* block_tables, int max_pages, hipStream_t st) {
  if (B < 1 || target < 1 || n_items < B || (block_tables && max_pages < 1)) return -1;
  hipLaunchKernelGGL(paged_decode_items_kernel, dim3(1), dim3(1024), 0, st, context_lens, (DecodeItem*)items, (int2*)rows, B,
                     target, n_items, finer, block_tables, max_pages);
  return (int)hipGetLastError();
}

template <int D, bool FP8, int NW>
static int launch_paged_decode_walk(const void* q, const void* kcache, const void* vcache, const int* block_tables,
                                    const int* context_lens, const void* items, int n_items, void* out, float* part_o,
                                    float* part_ml, int* arrived, int Hq, int Hkv, int max_pages, float scale_log2,
                                    int q_stride, hipStream_t st) {
  const size_t lds = (size_t)(NW * (Hq / Hkv) * (D + 4) + 2 * NW * 16) * sizeof(float);
  if (lds > 65536) {  // large groups: above the default limit
    static bool attr_set = false;
    if (!attr_set) {
      HIP_RET(hipFuncSetAttribute((const void*)paged_decode_walk_kernel<D, FP8, NW>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)((NW * 16 * (D + 4) + 2 * NW * 16) * sizeof(float))));
      attr_set = true;
    }
  }
  hipLaunchKernelGGL((paged_decode_walk_kernel<D, FP8, NW>), dim3(n_items * Hkv), dim3(64 * NW), lds, st, (const bf16_t*)q, kcache,
                     vcache, block_tables, context_lens, (const DecodeItem*)items, (bf16_t*)out, part_o, part_ml, arrived,
                     Hq, Hkv, Hq / Hkv, reciprocal((long)n_items * Hkv, Hkv), max_pages, scale_log2, q_stride);
  return (int)hipGetLastError();
}

// Decode attention over the items that areal_paged_decode_items made of the same context lengths. arrived null: the partial results of
// rows with several are left in part_o and part_ml for the kernel that follows, and `out` is written for the others only.
extern "C" int areal_paged_decode_walk(const void* q, const void* kcache, const void* vcache, const int* block_tables,
                                       const int* context_lens, const void* items, int n_items, void* out, float* part_o,
                                       float* part_ml, int* arrived, int Hq, int Hkv, int D, int max_pages,
                                       float softmax_scale, int q_stride, int fp8, hipStream_t st) {
  if (n_items == 0) return 0;
  if (Hq % Hkv != 0 || Hq / Hkv > 16) return -1;
  if (D != 128 && D != 64 && D != 256) return -2;
  const float scale_log2 = softmax_scale * 1.4426950408889634f;
#define PD(DD, F8, NW)                                                                                                  \
  return launch_paged_decode_walk<DD, F8, NW>(q, kcache, vcache, block_tables, context_lens, items, n_items, out, part_o, \
                                              part_ml, arrived, Hq, Hkv, max_pages, scale_log2, q_stride, st)
  if (D == 256) { if (fp8) PD(256, true, 4); else PD(256, false, 4); }
  if (D == 128) { if (fp8) PD(128, true, 8); else PD(128, false, 8); }
  if (fp8) PD(64, true, 8);
  PD(64, false, 8);
#undef PD
}

// ----------------------------------------------------------------------------------
// Fused RoPE + KV-cache write. qkv: [T, Hq + 2*Hkv, D] (q heads, k heads, v heads).
// Rotates q and k in place (half-split layout) and scatters k / v of every token into
// the paged caches at slot_mapping[t] (= page * 32 + offset; negative = skip the write).
// grid: T blocks; block: 256 threads.
// ----------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void rope_cache_write_kernel(
    bf16_t* __restrict__ qkv, const int* __restrict__ pos, const int64_t* __restrict__ slots,
    const float* __restrict__ cos_t, const float* __restrict__ sin_t, void* __restrict__ kcache,
    void* __restrict__ vcache, int Hq, int Hkv, int D, int max_pos, int do_rope, int fp8) {
  const int t = blockIdx.x;
  const int half = D >> 1;
  const int lph = half >> 3;  // lanes per head for the rotation
  int p = pos[t];
  p = p < 0 ? 0 : (p >= max_pos ? max_pos - 1 : p);
  bf16_t* row = qkv + (size_t)t * (Hq + 2 * Hkv) * D;
  const int64_t slot = slots ? slots[t] : -1;
  const int64_t page = slot >= 0 ? slot / PAGE : 0;
  const int off = slot >= 0 ? (int)(slot % PAGE) : 0;
  // phase 1: rotate q and k heads; k results go to the cache too
  const int nrot = (Hq + Hkv) * lph;
  for (int i = threadIdx.x; i < nrot; i += blockDim.x) {
    const int head = i / lph, sub = i % lph;
    bf16_t* base = row + (size_t)head * D + sub * 8;
    bf16x8 lo = ld8(base), hi = ld8(base + half);
    if (do_rope) {
      const float* cp = cos_t + (size_t)p * half + sub * 8;
      const float* sp = sin_t + (size_t)p * half + sub * 8;
      bf16x8 olo, ohi;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float a = bf2f(lo[j]), bb = bf2f(hi[j]);
        olo[j] = f2bf(a * cp[j] - bb * sp[j]);
        ohi[j] = f2bf(bb * cp[j] + a * sp[j]);
      }
      lo = olo; hi = ohi;
      st8(base, lo);
      st8(base + half, hi);
    }
    if (head >= Hq && slot >= 0) {
      const int kh = head - Hq;
      const size_t kd = (((size_t)page * Hkv + kh) * PAGE + off) * D + sub * 8;
      st8_cache(kcache, kd, lo, fp8);
      st8_cache(kcache, kd + half, hi, fp8);
    }
  }
  // phase 2: v heads -> transposed cache (scattered element stores, one page row apart)
  if (slot >= 0) {
    const bf16_t* vrow = row + (size_t)(Hq + Hkv) * D;
    for (int i = threadIdx.x; i < Hkv * D; i += blockDim.x) {
      const int vh = i / D, d = i % D;
      st1_cache(vcache, (((size_t)page * Hkv + vh) * D + d) * PAGE + off, bf2f(vrow[i]), fp8);
    }
  }
}

// The same for many tokens: 32 of them a workgroup. Tokens that follow each other in a prompt follow each other in a page, and
// eight of them from a multiple of eight on are one 16-byte store of a V channel instead of eight 2-byte stores to eight places of a
// 64-byte line (what bounded the kernel above, beside its idle threads). A workgroup writes the eights that start with one of its
// tokens; tokens of no whole eight (ends of prompts, rows in any order) go one by one. us of the two, prompts of 64 to 1216 tokens, 12
// heads on 2 of 128, 2048 / 4096 / 15600 / 32768 tokens: 8.9 / 12.9 / 46 / 91 and 11.4 / 12.5 / 36 / 68 (on an fp8 cache 7.7 / 11.1 / 38 /
// 72 and 11.9 / 12.9 / 34 / 66); 32 on 4 14 / 31 / 99 / 206 and 20 / 33 / 77 / 153; 14 on 2 of 64 6.3 / 8.9 / 27 / 58 and 7.7 / 9.0 / 21 / 41.
constexpr int RC_TOK = 32, RC_MIN_TOKENS = 8192, RC_THREADS = 1024;
__global__ __launch_bounds__(RC_THREADS) void rope_cache_write_many_kernel(
    bf16_t* __restrict__ qkv, const int* __restrict__ pos, const int64_t* __restrict__ slots,
    const float* __restrict__ cos_t, const float* __restrict__ sin_t, void* __restrict__ kcache,
    void* __restrict__ vcache, int T, int Hq, int Hkv, int D, int max_pos, int do_rope, int fp8) {
  extern __shared__ __attribute__((aligned(16))) bf16_t vbuf[];  // [RC_TOK + 7][Hkv D]: values of the tokens and of the seven behind
  __shared__ int64_t slot_of[RC_TOK + 14];                       // of tokens t0 - 7 ... ; -1: none
  __shared__ int run_at[RC_TOK / 8 + 1], n_runs;                 // first tokens (from t0) of the whole eights
  __shared__ int lone[RC_TOK], n_lone;
  const int t0 = blockIdx.x * RC_TOK, n = min(RC_TOK, T - t0), half = D >> 1, lph = half >> 3, W = Hkv * D, row_len = (Hq + 2 * Hkv) * D;
  if (threadIdx.x < RC_TOK + 14) {
    const int t = t0 - 7 + (int)threadIdx.x;
    slot_of[threadIdx.x] = t >= 0 && t < T ? slots[t] : -1;
  }
  if (threadIdx.x == 0) n_runs = n_lone = 0;
  for (int i = threadIdx.x; i < (RC_TOK + 7) * (W >> 3); i += RC_THREADS) {
    const int r = i / (W >> 3), ch = i - r * (W >> 3);
    if (t0 + r < T) st8(vbuf + r * W + ch * 8, ld8(qkv + (size_t)(t0 + r) * row_len + (Hq + Hkv) * D + ch * 8));
  }
  __syncthreads();
  if ((int)threadIdx.x < n) {  // whole eight that token `threadIdx.x` belongs to
    const int64_t s = slot_of[threadIdx.x + 7];
    if (s >= 0) {
      const int64_t first = s & ~7ll;
      const int at = (int)threadIdx.x + 7 - (int)(s - first);  // its place in slot_of, if the tokens before it are its neighbours
      bool whole = true;
      for (int j = 0; j < 8; ++j) whole = whole && slot_of[at + j] == first + j;
      if (!whole) lone[atomicAdd(&n_lone, 1)] = threadIdx.x;
      else if (s == first) run_at[atomicAdd(&n_runs, 1)] = threadIdx.x;
    }
  }
  const int heads = Hq + Hkv;
  for (int i = threadIdx.x; i < n * heads * lph; i += RC_THREADS) {
    const int sub = i % lph, rest = i / lph, head = rest % heads, r = rest / heads;
    const int64_t slot = slot_of[r + 7];
    bf16_t* base = qkv + (size_t)(t0 + r) * row_len + (size_t)head * D + sub * 8;
    bf16x8 lo = ld8(base), hi = ld8(base + half);
    if (do_rope) {
      int p = pos[t0 + r];
      p = p < 0 ? 0 : (p >= max_pos ? max_pos - 1 : p);
      const f32x4* cp = reinterpret_cast<const f32x4*>(cos_t + (size_t)p * half + sub * 8);
      const f32x4* sp = reinterpret_cast<const f32x4*>(sin_t + (size_t)p * half + sub * 8);
      bf16x8 olo, ohi;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float a = bf2f(lo[j]), bb = bf2f(hi[j]), c = cp[j >> 2][j & 3], sn = sp[j >> 2][j & 3];
        olo[j] = f2bf(a * c - bb * sn);
        ohi[j] = f2bf(bb * c + a * sn);
      }
      lo = olo; hi = ohi;
      st8(base, lo);
      st8(base + half, hi);
    }
    if (head >= Hq && slot >= 0) {
      const size_t kd = (((size_t)(slot / PAGE) * Hkv + head - Hq) * PAGE + slot % PAGE) * D + sub * 8;
      st8_cache(kcache, kd, lo, fp8);
      st8_cache(kcache, kd + half, hi, fp8);
    }
  }
  __syncthreads();
  // eights of one page beside each other: neighbouring lanes fill a channel's 64 bytes
  for (int i = threadIdx.x; i < n_runs * W; i += RC_THREADS) {
    const int r = run_at[i % n_runs], ch = i / n_runs, vh = ch / D, d = ch - vh * D;
    const int64_t slot = slot_of[r + 7];
    bf16x8 v;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = vbuf[(r + j) * W + ch];
    st8_cache(vcache, (((size_t)(slot / PAGE) * Hkv + vh) * D + d) * PAGE + slot % PAGE, v, fp8);
  }
  for (int i = threadIdx.x; i < n_lone * W; i += RC_THREADS) {
    const int r = lone[i / W], ch = i % W, vh = ch / D, d = ch - vh * D;
    const int64_t slot = slot_of[r + 7];
    st1_cache(vcache, (((size_t)(slot / PAGE) * Hkv + vh) * D + d) * PAGE + slot % PAGE, bf2f(vbuf[r * W + ch]), fp8);
  }
}

extern "C" int areal_rope_cache_write(void* qkv, const int* pos, const int64_t* slots,
                                      const float* cos_t, const float* sin_t, void* kcache,
                                      void* vcache, int T, int Hq, int Hkv, int D, int max_pos,
                                      int do_rope, int fp8, hipStream_t st) {
  if (T == 0) return 0;
  if (D % 16 != 0) return -1;
  const size_t lds = (size_t)(RC_TOK + 7) * Hkv * D * sizeof(bf16_t);
  // (60 KB beside the lists: what a launch may take without asking, two workgroups of 1024 threads a CU. V rows of more than 768 values, such as
  // 8 heads of 128, would leave one workgroup a CU, which was not measured: they keep a workgroup a token.)
  if (slots && T >= RC_MIN_TOKENS && lds <= 60 * 1024) {
    hipLaunchKernelGGL(rope_cache_write_many_kernel, dim3((T + RC_TOK - 1) / RC_TOK), dim3(RC_THREADS), lds, st, (bf16_t*)qkv, pos, slots,
                       cos_t, sin_t, kcache, vcache, T, Hq, Hkv, D, max_pos, do_rope, fp8);
    return (int)hipGetLastError();
  }
  hipLaunchKernelGGL(rope_cache_write_kernel, dim3(T), dim3(256), 0, st, (bf16_t*)qkv, pos, slots,
                     cos_t, sin_t, kcache, vcache, Hq, Hkv, D, max_pos, do_rope, fp8);
  return (int)hipGetLastError();
}

// Gather cached K/V of token slots back into contiguous [N, Hkv, D] tensors (used when a
// request extends a cached prefix: the prefix K/V are read from pages, the new tokens are
// appended, and the varlen flash kernel runs over the concatenation).
__global__ __launch_bounds__(256) void cache_gather_kernel(const void* __restrict__ kcache,
                                                           const void* __restrict__ vcache,
                                                           const int64_t* __restrict__ slots,
                                                           bf16_t* __restrict__ k_out,
                                                           bf16_t* __restrict__ v_out, int Hkv, int D,
                                                           int64_t out_stride, int fp8) {
  const int t = blockIdx.x;
  const int64_t slot = slots[t];
  const int64_t page = slot / PAGE;
  const int off = (int)(slot % PAGE);
  for (int i = threadIdx.x; i < Hkv * D; i += blockDim.x) {
    const int hh = i / D, d = i % D;
    const size_t ki = (((size_t)page * Hkv + hh) * PAGE + off) * D + d;
    const size_t vi = (((size_t)page * Hkv + hh) * D + d) * PAGE + off;
    if (fp8) {
      k_out[(size_t)t * out_stride + i] = f2bf(fp82f(reinterpret_cast<const fp8_t*>(kcache)[ki]));
      v_out[(size_t)t * out_stride + i] = f2bf(fp82f(reinterpret_cast<const fp8_t*>(vcache)[vi]));
    } else {
      k_out[(size_t)t * out_stride + i] = reinterpret_cast<const bf16_t*>(kcache)[ki];
      v_out[(size_t)t * out_stride + i] = reinterpret_cast<const bf16_t*>(vcache)[vi];
    }
  }
}

extern "C" int areal_cache_gather(const void* kcache, const void* vcache, const int64_t* slots,
                                  void* k_out, void* v_out, int N, int Hkv, int D, int64_t out_stride,
                                  int fp8, hipStream_t st) {
  if (N == 0) return 0;
  hipLaunchKernelGGL(cache_gather_kernel, dim3(N), dim3(256), 0, st, kcache, vcache, slots, (bf16_t*)k_out,
                     (bf16_t*)v_out, Hkv, D, out_stride, fp8);
  return (int)hipGetLastError();
}

// Copy whole pages (all layers share the same page ids): used for copy-on-write of a
// partially filled shared prefix page. kcache/vcache: [num_pages, page_elems].
__global__ void page_copy_kernel(bf16_t* __restrict__ cache, const int64_t* __restrict__ src,
                                 const int64_t* __restrict__ dst, int64_t page_elems) {
  const int64_t s = src[blockIdx.x], d = dst[blockIdx.x];
  for (int64_t i = threadIdx.x * 8; i < page_elems; i += (int64_t)blockDim.x * 8)
    st8(cache + d * page_elems + i, ld8(cache + s * page_elems + i));
}

extern "C" int areal_page_copy(void* cache, const int64_t* src, const int64_t* dst, int n,
                               int64_t page_elems, hipStream_t st) {
  if (n == 0) return 0;
  if (page_elems % 8 != 0) return -1;
  hipLaunchKernelGGL(page_copy_kernel, dim3(n), dim3(256), 0, st, (bf16_t*)cache, src, dst,
                     page_elems);
  return (int)hipGetLastError();
}

// Device-side bookkeeping between consecutive decode steps of one captured graph:
// feed the sampled token back, advance position / context length and derive the slot
// of the next token from the block table. Rows with active[b] == 0 are left untouched.
__global__ void advance_step_kernel(const int64_t* __restrict__ sampled, int64_t* __restrict__ input_ids,
                                    int* __restrict__ positions, int* __restrict__ context_lens,
                                    int64_t* __restrict__ slots, const int* __restrict__ block_tables,
                                    const int* __restrict__ active, int B, int max_pages) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  if (active && !active[b]) return;
  input_ids[b] = sampled[b];
  const int np = positions[b] + 1;
  positions[b] = np;
  context_lens[b] = np + 1;
  const int pg = np / PAGE;
  slots[b] = pg < max_pages ? (int64_t)block_tables[(size_t)b * max_pages + pg] * PAGE + np % PAGE : -1;
}

extern "C" int areal_advance_step(const int64_t* sampled, int64_t* input_ids, int* positions,
                                  int* context_lens, int64_t* slots, const int* block_tables,
                                  const int* active, int B, int max_pages, hipStream_t st) {
  if (B == 0) return 0;
  hipLaunchKernelGGL(advance_step_kernel, dim3((B + 255) / 256), dim3(256), 0, st, sampled, input_ids,
                     positions, context_lens, slots, block_tables, active, B, max_pages);
  return (int)hipGetLastError();
}


// ---------------------------------------------------------------------------------------------------
// Device-side bookkeeping of a multi-step decode plan with early exit.
//
// Per row: `active` (1 while the request still generates), `remaining` (tokens it may still produce:
// max_new_tokens and the context cap), `min_remaining` (tokens before stop ids count), `stop_ids`
// [B, n_stop] (-1 padded). After every sampled token the row either advances (next input token, position,
// context length, KV slot from the page table) or retires: no further KV writes (slot -1), attention over
// a single token (context length 1), sampler skipped. The host applies the same rules to the tokens it
// gets back, so both sides agree on where a request ends.
__global__ void decode_advance_kernel(const int64_t* __restrict__ sampled, int64_t* __restrict__ input_ids,
                                      int* __restrict__ positions, int* __restrict__ context_lens,
                                      int64_t* __restrict__ slots, const int* __restrict__ block_tables,
                                      int* __restrict__ active, int* __restrict__ remaining,
                                      int* __restrict__ min_remaining, const int* __restrict__ stop_ids,
                                      int n_stop, int B, int max_pages) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B || !active[b]) return;
  const int64_t tok = sampled[b];
  const int rem = remaining[b] - 1;
  const int mrem = min_remaining[b] > 0 ? min_remaining[b] - 1 : 0;
  remaining[b] = rem;
  min_remaining[b] = mrem;
  bool stop = rem <= 0;
  if (!stop && mrem == 0) {
    // stop ids count once min_new_tokens have been produced INCLUDING this token
    for (int j = 0; j < n_stop; ++j) stop |= stop_ids[(size_t)b * n_stop + j] == (int)tok;
  }
  if (stop) {
    active[b] = 0;
    slots[b] = -1;
    context_lens[b] = 1;
    return;
  }
  input_ids[b] = tok;
  const int np = positions[b] + 1;
  positions[b] = np;
  context_lens[b] = np + 1;
  const int pg = np / PAGE;
  slots[b] = pg < max_pages ? (int64_t)block_tables[(size_t)b * max_pages + pg] * PAGE + np % PAGE : -1;
}

// Start of a decode plan that continues the previous one on the same rows: rows whose request ended on
// the host (`kill`) retire, and live rows re-derive their KV slot from the refreshed page table.
__global__ void decode_begin_kernel(const int* __restrict__ kill, int* __restrict__ active,
                                    const int* __restrict__ positions, int* __restrict__ context_lens,
                                    int64_t* __restrict__ slots, const int* __restrict__ block_tables, int B,
                                    int max_pages) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  if (kill[b]) active[b] = 0;
  if (!active[b]) {
    slots[b] = -1;
    context_lens[b] = 1;
    return;
  }
  const int np = positions[b];
  const int pg = np / PAGE;
  slots[b] = pg < max_pages ? (int64_t)block_tables[(size_t)b * max_pages + pg] * PAGE + np % PAGE : -1;
}

extern "C" int areal_decode_advance(const int64_t* sampled, int64_t* input_ids, int* positions,
                                    int* context_lens, int64_t* slots, const int* block_tables, int* active,
                                    int* remaining, int* min_remaining, const int* stop_ids, int n_stop, int B,
                                    int max_pages, hipStream_t st) {
  if (B == 0) return 0;
  hipLaunchKernelGGL(decode_advance_kernel, dim3((B + 255) / 256), dim3(256), 0, st, sampled, input_ids,
                     positions, context_lens, slots, block_tables, active, remaining, min_remaining, stop_ids,
                     n_stop, B, max_pages);
  return (int)hipGetLastError();
}

extern "C" int areal_decode_begin(const int* kill, int* active, const int* positions, int* context_lens,
                                  int64_t* slots, const int* block_tables, int B, int max_pages,
                                  hipStream_t st) {
  if (B == 0) return 0;
  hipLaunchKernelGGL(decode_begin_kernel, dim3((B + 255) / 256), dim3(256), 0, st, kill, active, positions,
                     context_lens, slots, block_tables, B, max_pages);
  return (int)hipGetLastError();
}
