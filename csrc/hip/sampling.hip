// Fused temperature / top-k / top-p sampling with log-prob output for gfx950.
//
// One 1024-thread block per batch row. Replaces the torch sort/cumsum/topk logits
// warpers + Categorical sampling of the reference's native generator
// (realhf/impl/model/utils/logits_warper.py:52-125, 207-225;
// realhf/impl/model/nn/real_llm_generate.py:30-146) and SGLang's sampler.
//
//  * greedy (temperature == 0): arg-max.
//  * unfiltered (top_k >= V and top_p >= 1): Gumbel-max over z = logit / T, in the same single pass
//    over the row (16-byte loads) that accumulates the running max / sum-exp for the log-prob.
//  * filtered: thresholds for top-k (k-th largest z) and top-p (smallest set whose mass
//    reaches top_p of the top-k mass) are found by histograms over z (integer sums: order-independent),
//    then Gumbel-max runs over the surviving entries. No sort, no [B, V] temporaries.
//  * frequency / presence penalties: a request that asks for them owns a row of a token-count table
//    (`counts`, int16 [slots, count_ld]); its logits become logit - freq * count - pres * (count > 0)
//    before the temperature, in every pass, and the kernel bumps the count of the token it draws.
//  * rows flagged inactive (`active[row] == 0`: finished inside a multi-step decode plan) return at
//    once with token 0.
// The reported log-prob is log_softmax(adjusted logit / T)[token] over the FULL vocabulary (before
// top-k / top-p filtering); without penalties this is what the trainer recomputes.
// Randomness: Philox keyed by (seed, row, step) where `step` is read from device memory and
// can be bumped by the kernel itself, so a captured graph replays with fresh noise.
#include "common.hpp"

typedef short i16x8 __attribute__((ext_vector_type(8)));

struct ArgMax {
  float v;
  int i;
};
DEVINL ArgMax amax(ArgMax a, ArgMax b) {
  return (b.v > a.v || (b.v == a.v && b.i < a.i)) ? b : a;
}
DEVINL ArgMax block_argmax(ArgMax x, float* redv, int* redi) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    ArgMax y;
    y.v = __shfl_xor(x.v, o, 64);
    y.i = __shfl_xor(x.i, o, 64);
    x = amax(x, y);
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  __syncthreads();
  if (lane == 0) { redv[wid] = x.v; redi[wid] = x.i; }
  __syncthreads();
  ArgMax r;
  r.v = lane < nw ? redv[lane] : -INFINITY;
  r.i = lane < nw ? redi[lane] : 0x7fffffff;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    ArgMax y;
    y.v = __shfl_xor(r.v, o, 64);
    y.i = __shfl_xor(r.i, o, 64);
    r = amax(r, y);
  }
  return r;
}

template <typename T>
DEVINL float ldz(const T* p, int i) { return (float)p[i]; }

// 8 consecutive entries of a row as floats (one 16-byte load for bf16, two for fp32)
DEVINL void load8(const bf16_t* p, float* z) {
  const bf16x8 v = ld8(p);
#pragma unroll
  for (int j = 0; j < 8; ++j) z[j] = (float)v[j];
}
DEVINL void load8(const float* p, float* z) {
  const f32x4 a = *reinterpret_cast<const f32x4*>(p);
  const f32x4 b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
  for (int j = 0; j < 4; ++j) { z[j] = a[j]; z[4 + j] = b[j]; }
}

// One row of logits with its penalties: z_i = (logit_i - freq * count_i - pres * [count_i > 0]) / T.
template <typename T>
struct Row {
  const T* p;
  const int16_t* cnt;  // this request's token counts, or nullptr
  float freq, pres, inv_t;
  DEVINL float adjust(float x, int c) const { return x - freq * (float)c - (c > 0 ? pres : 0.f); }
  DEVINL float z1(int i) const {
    float x = ldz(p, i);
    if (cnt) x = adjust(x, cnt[i]);
    return x * inv_t;
  }
  // entries [i8, i8 + 8), i8 a multiple of 8 (16-byte loads of the logits and of the counts)
  DEVINL void z8(int i8, float* z) const {
    load8(p + i8, z);
    if (cnt) {
      const i16x8 c = *reinterpret_cast<const i16x8*>(cnt + i8);
#pragma unroll
      for (int j = 0; j < 8; ++j) z[j] = adjust(z[j], c[j]);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) z[j] *= inv_t;
  }
};

// f(i, z_i) over one row: vector loads over [0, V8), scalar loads over the tail [V8, V)
// (a thread's chunks are fetched four at a time: with one load in flight a pass over a 152k-entry row is a chain of
// ~19 memory round trips per thread)
template <typename T, typename F>
DEVINL void for_each_z(const Row<T>& r, int V, int V8, F f) {
  constexpr int PF = 4;
  const int stride = blockDim.x * 8;
  for (int base = threadIdx.x * 8; base < V8; base += stride * PF) {
    float zz[PF][8];
#pragma unroll
    for (int u = 0; u < PF; ++u)
      if (base + u * stride < V8) r.z8(base + u * stride, zz[u]);
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      const int i8 = base + u * stride;
      if (i8 >= V8) break;
#pragma unroll
      for (int j = 0; j < 8; ++j) f(i8 + j, zz[u][j]);
    }
  }
  for (int i = V8 + threadIdx.x; i < V; i += blockDim.x) f(i, r.z1(i));
}

// __logf of a positive, normal, finite number: the same bits without the scaling of subnormals and the test for infinities, 5
// instructions for 14. Both arguments below are such: 2^-24 .. 1 - 2^-24 and the negated logarithms of these. (sample_partial_kernel,
// 320 rows of 151936 at temperature 1: 84 -> 66 us, with the largest of eight keys found before their index is compared.)
DEVINL float log_normal(float x) {
  const float l = __builtin_amdgcn_logf(x), hi = 0x1.62e42ep-1f, lo = 0x1.efa39ep-25f;
  return fmaf(l, hi, fmaf(l, lo, fmaf(l, hi, -(l * hi))));
}
DEVINL float gumbel(uint32_t bits) { return -log_normal(-log_normal(u32_to_unit(bits) * 0.99999994f)); }

// ---------------------------------------------------------------------------------------------
// Thresholds of top-k and top-p: the largest entry t of a row with F(t) >= target, F(t) = number (MASS = false) or
// softmax mass relative to exp(-mx) (MASS = true) of the entries z >= t. A pass over the row sorts the entries of a
// bracket [lo, hi] into SEL_BINS bins of equal width (LDS atomics) and finds the bin that holds t; its entries are copied
// into LDS and split the same way until at most SEL_DIRECT are left, whose F are summed directly. What bounds it is
// vector instructions of the one workgroup that owns a row: a pass over 151936 entries takes 4 to 10 us however few
// bytes it reads, so the number of passes counts. Halving the bracket instead took five to ten passes over the row and
// some 25 block-wide sums after them. 24 rows of 151936 bf16 entries, before and now: top-p 0.95 of normal logits 246 and
// 132 us, of one dominant token 85 and 45; top-k 50 99 and 57, with top-p 0.9 160 and 86; 320 rows of the first 507 and 271.
// Counts and masses (fixed point, 2^-40) are integers: no result depends on the order in which atomics arrive, so
// replays and the ranks of a tensor-parallel group agree bit for bit. Entries more than SEL_RANGE below the maximum
// have no mass at this resolution.
constexpr int SEL_BINS = 1024;     // one per thread
constexpr int SEL_CAP = 4096;      // entries of a bin that are copied into LDS (a fuller bin is split again from the row)
constexpr int SEL_DIRECT = 256;
constexpr float SEL_FIX = 1099511627776.f;  // 2^40
constexpr float SEL_RANGE = 28.f;

struct Select {
  unsigned long long mass[SEL_BINS];
  unsigned cnt[SEL_BINS];
  float cand[SEL_CAP], few[SEL_DIRECT];
  unsigned long long part[16], above;
  int bin, n;
  unsigned bin_n;
};

// monotone in z: the bins are an ordered partition of [lo, hi] (no contraction with the product that made z, so that
// every pass puts an entry into the same bin)
DEVINL int sel_bin(float z, float lo, float scale) {
#pragma clang fp contract(off)
  const float d = z - lo;
  return min(SEL_BINS - 1, (int)(d * scale));
}

DEVINL unsigned long long sel_mass(float z, float mx) {
#pragma clang fp contract(off)
  const float d = z - mx;
  return (unsigned long long)(__expf(d) * SEL_FIX);
}

// The bin of [lo, hi] in which F reaches target (S.bin, -1: none), F above it (S.above; of everything if none) and its
// number of entries (S.bin_n). each(f) calls f(z) for every entry, over the whole block.
template <bool MASS, typename E>
DEVINL void select_bin(Select& S, E each, float lo, float hi, float scale, float mx, unsigned long long above,
                       unsigned long long target) {
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  __syncthreads();
  S.cnt[tid] = 0u;
  if (MASS) S.mass[tid] = 0ull;
  if (tid == 0) S.bin = -1;
  __syncthreads();
  each([&](float z) {
    if (z >= lo && z <= hi) {
      const int b = sel_bin(z, lo, scale);
      atomicAdd(&S.cnt[b], 1u);
      if (MASS) atomicAdd(&S.mass[b], sel_mass(z, mx));
    }
  });
  __syncthreads();
  const int b = SEL_BINS - 1 - tid;  // from the top bin down
  const unsigned c = S.cnt[b];
  const unsigned long long w = MASS ? S.mass[b] : (unsigned long long)c;
  unsigned long long run = w;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned long long y = __shfl_up(run, o, 64);
    if (lane >= o) run += y;
  }
  if (lane == 63) S.part[wid] = run;
  __syncthreads();
  run += above;
  for (int i = 0; i < wid; ++i) run += S.part[i];
  if (run >= target && run - w < target) {  // at most one bin
    S.bin = b;
    S.above = run - w;
    S.bin_n = c;
  }
  __syncthreads();
  if (S.bin < 0 && tid == SEL_BINS - 1) S.above = run;
  __syncthreads();
}

// row(f): f(z) for every entry, over the whole block. floor: entries below it do not count (the top-k threshold, or -inf);
// mn, mx: smallest and largest finite entry. Returns floor where even all entries fall short of the target.
template <bool MASS, typename E>
DEVINL float select_threshold(Select& S, E row, float floor, float mn, float mx, float target_f, float* red) {
  if (!(mx < INFINITY) || !(mx > -INFINITY) || target_f != target_f) return floor;
  const int tid = threadIdx.x;
  const float bottom = fmaxf(floor, mn);
  const double tf = MASS ? ceil((double)target_f * (double)SEL_FIX) : (double)target_f;
  const unsigned long long target = tf < 1. ? 1ull : (unsigned long long)tf;
  unsigned long long above = 0ull;
  float lo = fmaxf(bottom, mx - SEL_RANGE), hi = mx, scale = 0.f;
  int n = 0;
  for (int round = 0;; ++round) {
    if (round == 8) return lo;
    scale = hi > lo ? (float)SEL_BINS / (hi - lo) : 0.f;
    if (!(scale < INFINITY)) scale = 0.f;  // a bracket of denormal width: one bin
    select_bin<MASS>(S, row, lo, hi, scale, mx, above, target);
    above = S.above;
    const int bin = S.bin;
    if (bin < 0) {
      if (lo <= bottom) return floor;
      hi = nextafterf(lo, -INFINITY);
      lo = bottom;
      continue;
    }
    if (scale == 0.f) return lo;
    n = (int)S.bin_n;
    if (n <= SEL_CAP) {
      __syncthreads();
      if (tid == 0) S.n = 0;
      __syncthreads();
      row([&](float z) {
        if (z >= lo && z <= hi && sel_bin(z, lo, scale) == bin) {
          const int pos = atomicAdd(&S.n, 1);
          if (pos < SEL_CAP) S.cand[pos] = z;
        }
      });
      __syncthreads();
      break;
    }
    float l = INFINITY, h = -INFINITY;
    row([&](float z) {
      if (z >= lo && z <= hi && sel_bin(z, lo, scale) == bin) {
        l = fminf(l, z);
        h = fmaxf(h, z);
      }
    });
    lo = -block_max(-l, red);
    hi = block_max(h, red);
  }
  // ---- the n entries of the bin, in LDS
  auto list = [&](auto f) __attribute__((always_inline)) { for (int i = tid; i < n; i += SEL_BINS) f(S.cand[i]); };
  const float* last = S.cand;
  int m = n;
  if (n > SEL_DIRECT) {
    float l = INFINITY, h = -INFINITY;
    list([&](float z) { l = fminf(l, z); h = fmaxf(h, z); });
    lo = -block_max(-l, red);
    hi = block_max(h, red);
    for (int round = 0;; ++round) {
      scale = hi > lo ? (float)SEL_BINS / (hi - lo) : 0.f;
      if (round == 8 || scale == 0.f || !(scale < INFINITY)) return lo;
      select_bin<MASS>(S, list, lo, hi, scale, mx, above, target);
      above = S.above;
      const int bin = S.bin;
      m = (int)S.bin_n;
      if (m <= SEL_DIRECT) {
        __syncthreads();
        if (tid == 0) S.n = 0;
        __syncthreads();
        list([&](float z) {
          if (z >= lo && z <= hi && sel_bin(z, lo, scale) == bin) {
            const int pos = atomicAdd(&S.n, 1);
            if (pos < SEL_DIRECT) S.few[pos] = z;
          }
        });
        __syncthreads();
        last = S.few;
        break;
      }
      l = INFINITY, h = -INFINITY;
      list([&](float z) {
        if (z >= lo && z <= hi && sel_bin(z, lo, scale) == bin) {
          l = fminf(l, z);
          h = fmaxf(h, z);
        }
      });
      lo = -block_max(-l, red);
      hi = block_max(h, red);
    }
  }
  float t = -INFINITY;
  if (tid < m) S.mass[tid] = MASS ? sel_mass(last[tid], mx) : 1ull;
  __syncthreads();
  if (tid < m) {
    const float z = last[tid];
    unsigned long long f = above;
    for (int i = 0; i < m; ++i) f += last[i] >= z ? S.mass[i] : 0ull;
    if (f >= target) t = z;
  }
  t = block_max(t, red);
  return t > -INFINITY ? t : lo;
}

// ---------------------------------------------------------------------------------------------
// Filtered rows, first part: S workgroups a row, each with a slice of it: the slice's maximum, minimum and sum of exponentials.
// With a small top-k what the workgroup that owns the row then still needs of its 152k entries are those that can be among the
// k largest, so every slice also hands on a superset of its own k largest entries (the bins of its histogram from the k-th
// largest's on): seven passes of one workgroup over the row become two of S workgroups over a slice and work on a few
// hundred entries. us of one part and of two, top-k 50 with top-p 0.95, 1 / 64 / 200 / 320 rows: 151936 bf16 entries 83 / 86 / 108 /
// 191 and 31 / 35 / 57 / 87, 32000 of them 33 / 35 / 35 / 66 and 25 / 26 / 29 / 52; 50257, whose rows start off the 16-byte grid and
// are walked entry by entry, 42 / 78 / 79 / 161 and 27 / 32 / 54 / 81.
// ws: [B][S][SLICE_WORDS] words: {max, sum of exp(z - max), number of entries (-1: none or too many, the row's own passes find
// the set), min}, entries, their places; behind them the step (the second part's first workgroup counts it on, so the others
// read it here).
constexpr int TOPK_MAX = 128, TOPK_CAP = 256, SLICE_WORDS = 4 + 2 * TOPK_CAP, SLICES = SEL_CAP / TOPK_CAP, SLICE_THREADS = 512;

// Whether the row's slices do anything: with a small top-k, or where there are enough of them to shorten the first pass. us of
// one part and of two, top-p 0.95 alone, 8 / 4 / 2 slices (64 / 128 / 256 rows): 151936 bf16 entries 127 / 138 / 140 and 124 / 132 /
// 140, 65536 fp32 69 / 70 / 84 and 69 / 74 / 86, 32000 fp32 41 / 42 / 44 and 43 / 43 / 50.
DEVINL bool row_sliced(int k, int V, int S) { return (k >= 1 && k < V && k <= TOPK_MAX) || S >= 8; }

template <typename T>
__global__ __launch_bounds__(SLICE_THREADS) void sample_slice_kernel(
    const T* __restrict__ logits, int64_t ld, int V, const float* __restrict__ temperature, const int* __restrict__ top_k,
    const float* __restrict__ top_p, const int64_t* __restrict__ step_ptr, const int* __restrict__ active,
    const int16_t* __restrict__ counts, int64_t count_ld, const int* __restrict__ count_slot,
    const float* __restrict__ freq_pen, const float* __restrict__ pres_pen, float* __restrict__ ws, int S) {
  constexpr int NT = SLICE_THREADS, BINS = 1024, PER = BINS / NT;
  __shared__ float red[16];
  __shared__ unsigned hist[BINS], part[NT / 64];
  __shared__ int s_bin, s_above, s_n, s_pos;
  const int row = blockIdx.y, s = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  if (row == 0 && s == 0 && tid == 0 && step_ptr)
    *reinterpret_cast<int64_t*>(ws + (size_t)gridDim.y * S * SLICE_WORDS) = step_ptr[0];
  if (active && !active[row]) return;
  const float temp = temperature ? temperature[row] : 1.f;
  const int k = top_k ? top_k[row] : V;
  const bool limited = k >= 1 && k < V;
  if (temp <= 0.f || !(limited || (top_p && top_p[row] < 1.f)) || !row_sliced(k, V, S)) return;
  const T* p = logits + (size_t)row * ld;
  const int V8 = (reinterpret_cast<uintptr_t>(p) & 15) == 0 ? (V & ~7) : 0;
  const int slot = (counts && count_slot) ? count_slot[row] : -1;
  Row<T> R;
  R.p = p;
  R.cnt = slot >= 0 ? counts + (size_t)slot * count_ld : nullptr;
  R.freq = R.cnt && freq_pen ? freq_pen[row] : 0.f;
  R.pres = R.cnt && pres_pen ? pres_pen[row] : 0.f;
  R.inv_t = 1.f / temp;
  const int chunks = V8 >> 3, per = (chunks + S - 1) / S;
  const int first = min(chunks, s * per) * 8, end = min(chunks, (s + 1) * per) * 8;
  // f8(i, z) over groups of 8 entries of the slice, f1(i, z_i) over those behind the last whole group (or over the whole row
  // when it is not 16-byte aligned)
  auto walk = [&](auto f8, auto f1) __attribute__((always_inline)) {
    constexpr int PF = 4;
    for (int base = first + tid * 8; base < end; base += NT * 8 * PF) {
      float zz[PF][8];
#pragma unroll
      for (int u = 0; u < PF; ++u)
        if (base + u * NT * 8 < end) R.z8(base + u * NT * 8, zz[u]);
#pragma unroll
      for (int u = 0; u < PF; ++u) {
        const int i8 = base + u * NT * 8;
        if (i8 >= end) break;
        f8(i8, zz[u]);
      }
    }
    for (int i = V8 + s * NT + tid; i < V; i += S * NT) f1(i, R.z1(i));
  };
  auto each = [&](auto f) __attribute__((always_inline)) {
    walk([&](int i8, const float* z) {
#pragma unroll
      for (int j = 0; j < 8; ++j) f(i8 + j, z[j]);
    }, f);
  };
  float mx = -INFINITY, mn = INFINITY, se = 0.f;
  auto raise = [&](float m) {
    if (m > mx) {
      se *= __expf(mx - m);
      mx = m;
    }
  };
  walk([&](int, const float* z) {
    float m8 = -INFINITY;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      m8 = fmaxf(m8, z[j]);
      mn = fminf(mn, z[j] > -INFINITY ? z[j] : INFINITY);
    }
    raise(m8);
    if (mx > -INFINITY)
#pragma unroll
      for (int j = 0; j < 8; ++j) se += __expf(z[j] - mx);
  }, [&](int, float z) {
    mn = fminf(mn, z > -INFINITY ? z : INFINITY);
    raise(z);
    if (mx > -INFINITY) se += __expf(z - mx);
  });
  const float own = mx;  // this thread's largest entry
  const float mx_all = block_max(mx, red);
  mn = -block_max(-mn, red);
  se = block_sum(mx > -INFINITY ? se * __expf(mx - mx_all) : 0.f, red);
  mx = mx_all;
  float* o = ws + ((size_t)row * S + s) * SLICE_WORDS;
  // The bin of [lo, hi] from which on there are k entries, from the top down (s_bin, -1: fewer in all), their number in the bin
  // and above it; `above` entries lie above hi. fill(f): f(z) for every entry that counts
  float lo = mn, hi = mx, scale = 0.f;
  int bin = 0, above = 0;
  auto find = [&](auto fill) __attribute__((always_inline)) {
    scale = hi > lo ? (float)BINS / (hi - lo) : 0.f;
    if (!(scale < INFINITY)) scale = 0.f;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i) hist[i * NT + tid] = 0u;
    if (tid == 0) s_bin = -1;
    __syncthreads();
    fill([&](float z) {
      if (z >= lo && z <= hi) atomicAdd(&hist[sel_bin(z, lo, scale)], 1u);
    });
    __syncthreads();
    unsigned c[PER], sum = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) sum += c[i] = hist[BINS - 1 - (tid * PER + i)];
    unsigned run = sum;
#pragma unroll
    for (int of = 1; of < 64; of <<= 1) {
      const unsigned y = __shfl_up(run, of, 64);
      if (lane >= of) run += y;
    }
    if (lane == 63) part[wid] = run;
    __syncthreads();
    run += above - sum;
    for (int i = 0; i < wid; ++i) run += part[i];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if ((int)run < k && (int)(run + c[i]) >= k) {
        s_bin = BINS - 1 - (tid * PER + i);
        s_above = (int)run;
        s_n = (int)c[i];
      }
      run += c[i];
    }
    __syncthreads();
    bin = s_bin;
  };
  // Hands on the entries from the bin on (of a bracket that ends at the largest entry, or one that lies in such a bin); their number
  auto hand_on = [&]() __attribute__((always_inline)) {
    __syncthreads();
    if (tid == 0) s_pos = 0;
    __syncthreads();
    each([&](int i, float z) {
      if (z > hi || (z >= lo && sel_bin(z, lo, scale) >= bin)) {
        const int at = atomicAdd(&s_pos, 1);
        if (at < TOPK_CAP) {
          o[4 + at] = z;
          o[4 + TOPK_CAP + at] = __int_as_float(i);
        }
      }
    });
    __syncthreads();
    return s_pos;
  };
  int n = -1;  // entries handed on
  if (limited && k <= TOPK_MAX && mx < INFINITY) {
    if (!(mx > -INFINITY)) {
      n = 0;
    } else {
      // the k-th largest of the threads' largest entries is no larger than the k-th largest entry, and for entries in no
      // particular order not much smaller: a little over k of them reach it
      const float low = -block_max(own > -INFINITY ? -own : -INFINITY, red);
      lo = low;
      find([&](auto f) { if (own > -INFINITY) f(own); });
      if (bin < 0) {  // fewer threads than k have entries: all of them
        lo = mn;
        scale = 0.f;
        bin = 0;
      }
      n = hand_on();
      lo = mn;
      hi = mx;
      for (int round = 0; n > TOPK_CAP; ++round) {  // too many: the bin of the k-th largest entry itself
        find([&](auto f) { each([&](int, float z) { f(z); }); });
        if (bin < 0 || s_above + s_n <= TOPK_CAP) {
          bin = max(bin, 0);
          n = hand_on();
          break;
        }
        if (scale == 0.f || round == 6) break;
        above = s_above;
        float l = INFINITY, h = -INFINITY;
        each([&](int, float z) {
          if (z >= lo && z <= hi && sel_bin(z, lo, scale) == bin) {
            l = fminf(l, z);
            h = fmaxf(h, z);
          }
        });
        lo = -block_max(-l, red);
        hi = block_max(h, red);
      }
    }
  }
  if (tid == 0) {
    o[0] = mx;
    o[1] = se;
    o[2] = __int_as_float(n > TOPK_CAP ? -1 : n);
    o[3] = mn;
  }
}

// ws, S: what sample_slice_kernel has left (null: nothing; the rows' statistics are then a pass of this kernel's own, and step_ptr
// is not counted on)
template <typename T>
__global__ __launch_bounds__(1024) void sample_kernel(
    const T* __restrict__ logits, int64_t ld, int V, const float* __restrict__ temperature,
    const int* __restrict__ top_k, const float* __restrict__ top_p, uint64_t seed,
    int64_t* step_ptr, int64_t* __restrict__ out_tok,
    float* __restrict__ out_logp, const int* __restrict__ active, int16_t* __restrict__ counts,
    int64_t count_ld, const int* __restrict__ count_slot, const float* __restrict__ freq_pen,
    const float* __restrict__ pres_pen, const float* __restrict__ ws, int S, int bump_step) {
  __shared__ float red[16];
  __shared__ float redv[16];
  __shared__ int redi[16];
  __shared__ Select sel;
  __shared__ float list_z[SEL_CAP];
  __shared__ int list_i[SEL_CAP];
  const int row = blockIdx.x;
  const int64_t* step_at = ws ? reinterpret_cast<const int64_t*>(ws + (size_t)gridDim.x * S * SLICE_WORDS) : step_ptr;
  const uint64_t step = step_ptr ? (uint64_t)step_at[0] : 0;
  if (ws && step_ptr && bump_step && row == 0 && threadIdx.x == 0) step_ptr[0] = (int64_t)step + 1;
  if (active && !active[row]) {  // uniform over the block
    if (threadIdx.x == 0) {
      out_tok[row] = 0;
      if (out_logp) out_logp[row] = 0.f;
    }
    return;
  }
  const T* p = logits + (size_t)row * ld;
  const float temp = temperature ? temperature[row] : 1.f;
  const bool greedy = temp <= 0.f;
  const float inv_t = greedy ? 1.f : 1.f / temp;
  const int k = top_k ? top_k[row] : V;
  const float tp = top_p ? top_p[row] : 1.f;
  const bool filtered = !greedy && ((k < V && k >= 1) || tp < 1.f);
  // noise word of entry i: word i & 3 of the Philox block with counter ctr0 + i / 4
  const uint64_t ctr0 = step * (uint64_t)((V + 3) / 4);
  const int V8 = (reinterpret_cast<uintptr_t>(p) & 15) == 0 ? (V & ~7) : 0;
  const int slot = (counts && count_slot) ? count_slot[row] : -1;
  int16_t* cnt = slot >= 0 ? counts + (size_t)slot * count_ld : nullptr;  // count_ld is a multiple of 8
  Row<T> R;
  R.p = p;
  R.cnt = cnt;
  R.freq = cnt && freq_pen ? freq_pen[row] : 0.f;
  R.pres = cnt && pres_pen ? pres_pen[row] : 0.f;
  R.inv_t = inv_t;

  float mx = -INFINITY, mn = INFINITY, se = 0.f;
  const bool sliced = ws && filtered && row_sliced(k, V, S);
  bool listed = sliced;  // the slices have handed on all that can be drawn
  // A lane reads a slice's words and a wave copies its entries: one slice after the other they were a chain of up to 16 trips to
  // memory (24 rows of 151936 entries in 8 slices, top-k 50 with top-p 0.95: 34.0 us for both kernels, 30.8 now).
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int handed = 0;
  if (sliced) {
    f32x4 o = {-INFINITY, 0.f, 0.f, INFINITY};
    if (lane < S) o = *reinterpret_cast<const f32x4*>(ws + ((size_t)row * S + lane) * SLICE_WORDS);
    mx = o[0];
    mn = o[3];
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
      mx = fmaxf(mx, __shfl_xor(mx, d, 64));
      mn = fminf(mn, __shfl_xor(mn, d, 64));
    }
    handed = __float_as_int(o[2]);
    listed = !__any(handed < 0);
    const float scale = o[0] > -INFINITY ? __expf(o[0] - mx) : 0.f;
    for (int s = 0; s < S; ++s)  // in the order of the slices
      se += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(o[1]), s)) *
            __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(scale), s));
  }
  if (listed) {
    int n = 0;
    for (int s = 0; s < S; ++s) {
      const int c = __builtin_amdgcn_readlane(handed, s);
      if ((s & 15) == wid) {  // one of the block's 16 waves
        const float* o = ws + ((size_t)row * S + s) * SLICE_WORDS + 4;
        for (int i = lane; i < c; i += 64) {
          list_z[n + i] = o[i];
          list_i[n + i] = __float_as_int(o[TOPK_CAP + i]);
        }
      }
      n += c;
    }
    __syncthreads();
    auto list = [&](auto f) __attribute__((always_inline)) { for (int i = threadIdx.x; i < n; i += blockDim.x) f(list_z[i]); };
    mn = INFINITY;
    list([&](float z) { mn = fminf(mn, z); });
    mn = -block_max(-mn, red);
    float thr = select_threshold<false>(sel, list, -INFINITY, mn, mx, (float)k, red);
    if (tp < 1.f) {  // mass of the top-k set, the nucleus's reference: an integer, for the entries come in any order
      unsigned long long m = 0ull;
      list([&](float z) { m += z >= thr ? sel_mass(z, mx) : 0ull; });
#pragma unroll
      for (int of = 32; of > 0; of >>= 1) m += __shfl_xor(m, of, 64);
      __syncthreads();
      if ((threadIdx.x & 63) == 0) sel.part[threadIdx.x >> 6] = m;
      __syncthreads();
      m = 0ull;
      for (int w = 0; w < 16; ++w) m += sel.part[w];
      __syncthreads();
      thr = select_threshold<true>(sel, list, thr, mn, mx, tp * (float)((double)m / (double)SEL_FIX), red);
    }
    ArgMax best;
    best.v = -INFINITY;
    best.i = 0x7fffffff;
    for (int i = threadIdx.x; i < n; i += blockDim.x)
      if (list_z[i] >= thr) {
        ArgMax c;
        c.i = list_i[i];
        c.v = list_z[i] + gumbel(Philox::gen(seed, (uint64_t)row, ctr0 + (uint64_t)(c.i >> 2))[c.i & 3]);
        best = amax(best, c);
      }
    best = block_argmax(best, redv, redi);
    if (threadIdx.x == 0) {
      int tok = best.i;
      if (tok < 0 || tok >= V) tok = 0;
      out_tok[row] = tok;
      if (out_logp) out_logp[row] = R.z1(tok) - (mx + __logf(se));
      if (cnt && cnt[tok] < 32767) cnt[tok] += 1;
    }
    return;
  }

  // pass 1: running max / sum-exp (rescaled when the max moves) and min of z. Without filtering the
  // arg-max of z (+ Gumbel noise unless greedy) is taken in the same pass, so the row is read once.
  const bool pick_now = !filtered;
  const bool noise = !greedy;
  ArgMax best;
  best.v = -INFINITY;
  best.i = 0x7fffffff;
  // The row is walked in groups of PF chunks per thread whose loads are all issued before the first one is used: a
  // thread sees ~19 chunks of a 152k-entry row, and with one load in flight at a time the pass is a chain of that
  // many memory round trips (the per-entry noise and exponentials are cheap next to them).
  constexpr int PF = 4;
  if (!sliced) {
    for (int base = threadIdx.x * 8; base < V8; base += blockDim.x * 8 * PF) {
      float zz[PF][8];
#pragma unroll
      for (int u = 0; u < PF; ++u) {
        const int i8 = base + u * (int)blockDim.x * 8;
        if (i8 < V8) R.z8(i8, zz[u]);
      }
#pragma unroll
      for (int u = 0; u < PF; ++u) {
        const int i8 = base + u * (int)blockDim.x * 8;
        if (i8 >= V8) break;
        float* z = zz[u];
        float m8 = -INFINITY;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          m8 = fmaxf(m8, z[j]);
          mn = fminf(mn, z[j] > -INFINITY ? z[j] : INFINITY);
        }
        if (m8 > mx) {
          se *= __expf(mx - m8);
          mx = m8;
        }
        if (mx > -INFINITY) {
#pragma unroll
          for (int j = 0; j < 8; ++j) se += __expf(z[j] - mx);
        }
        if (pick_now) {
          u32x4 r0, r1;
          if (noise) {
            r0 = Philox::gen(seed, (uint64_t)row, ctr0 + (uint64_t)(i8 >> 2));
            r1 = Philox::gen(seed, (uint64_t)row, ctr0 + (uint64_t)(i8 >> 2) + 1);
          }
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            ArgMax c;
            c.v = noise ? z[j] + gumbel(j < 4 ? r0[j] : r1[j - 4]) : z[j];
            c.i = i8 + j;
            best = amax(best, c);
          }
        }
      }
    }
    for (int i = V8 + threadIdx.x; i < V; i += blockDim.x) {
      const float z = R.z1(i);
      mn = fminf(mn, z > -INFINITY ? z : INFINITY);
      if (z > mx) {
        se *= __expf(mx - z);
        mx = z;
      }
      if (mx > -INFINITY) se += __expf(z - mx);
      if (pick_now) {
        ArgMax c;
        c.v = z;
        c.i = i;
        if (noise) c.v += gumbel(Philox::gen(seed, (uint64_t)row, ctr0 + (uint64_t)(i >> 2))[i & 3]);
        best = amax(best, c);
      }
    }
    const float mx_all = block_max(mx, red);
    mn = -block_max(-mn, red);
    se = block_sum(mx > -INFINITY ? se * __expf(mx - mx_all) : 0.f, red);
    mx = mx_all;
  }
  const float lse = mx + __logf(se);

  if (filtered) {
    float thr = -INFINITY;
    float mass_k = se;  // mass (relative to exp(-mx)) of the top-k set
    auto all = [&](auto f) __attribute__((always_inline)) { for_each_z(R, V, V8, [&](int, float z) { f(z); }); };
    if (k < V && k >= 1) {
      thr = select_threshold<false>(sel, all, -INFINITY, mn, mx, (float)k, red);
      if (tp < 1.f) {  // the nucleus is taken inside the top-k set: its mass is the reference
        float mk = 0.f;
        for_each_z(R, V, V8, [&](int, float z) {
          if (z >= thr) mk += __expf(z - mx);
        });
        mass_k = block_sum(mk, red);
      }
    }
    if (tp < 1.f) thr = select_threshold<true>(sel, all, thr, mn, mx, tp * mass_k, red);
    // arg-max of z + Gumbel noise over the entries that survive the threshold. The noise block of four entries is made
    // once, and only where one of them survives: with a block per entry a nucleus of 100k entries took 33 us longer.
    for (int base = threadIdx.x * 8; base < V8; base += blockDim.x * 8 * PF) {
      float zz[PF][8];
#pragma unroll
      for (int u = 0; u < PF; ++u) {
        const int i8 = base + u * (int)blockDim.x * 8;
        if (i8 < V8) R.z8(i8, zz[u]);
      }
#pragma unroll
      for (int u = 0; u < PF; ++u) {
        const int i8 = base + u * (int)blockDim.x * 8;
        if (i8 >= V8) break;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float* z = zz[u] + 4 * h;
          if (fmaxf(fmaxf(z[0], z[1]), fmaxf(z[2], z[3])) >= thr) {
            const u32x4 r = Philox::gen(seed, (uint64_t)row, ctr0 + (uint64_t)(i8 >> 2) + h);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              ArgMax c;
              c.v = z[j] >= thr ? z[j] + gumbel(r[j]) : -INFINITY;
              c.i = z[j] >= thr ? i8 + 4 * h + j : 0x7fffffff;
              best = amax(best, c);
            }
          }
        }
      }
    }
    for (int i = V8 + threadIdx.x; i < V; i += blockDim.x) {
      const float z = R.z1(i);
      if (z >= thr) {
        ArgMax c;
        c.v = z + gumbel(Philox::gen(seed, (uint64_t)row, ctr0 + (uint64_t)(i >> 2))[i & 3]);
        c.i = i;
        best = amax(best, c);
      }
    }
  }
  best = block_argmax(best, redv, redi);
  if (threadIdx.x == 0) {
    int tok = best.i;
    if (tok < 0 || tok >= V) tok = 0;
    out_tok[row] = tok;
    if (out_logp) out_logp[row] = R.z1(tok) - lse;
    if (cnt && cnt[tok] < 32767) cnt[tok] += 1;
  }
}

// ---------------------------------------------------------------------------------------------
// Unfiltered sampling (no top-k / top-p anywhere in the batch) with every row split over `S` workgroups: one
// 1024-thread workgroup per row leaves a 384-row decode batch with 1.5 workgroups per CU, each walking 152k entries
// as a chain of dependent passes. Here S x B workgroups of 256 threads each reduce a slice of a row to
// (max, sum-exp relative to it, best perturbed value, its index); a one-wave-per-row kernel merges the slices,
// writes token and log-prob, bumps the token count and the step. The noise of entry i is the same Philox word as
// in the one-workgroup kernel, so both draw the SAME token; the log-prob differs by summation order only.
template <typename T>
__global__ __launch_bounds__(256) void sample_partial_kernel(
    const T* __restrict__ logits, int64_t ld, int V, const float* __restrict__ temperature, uint64_t seed,
    const int64_t* __restrict__ step_ptr, const int* __restrict__ active, const int16_t* __restrict__ counts,
    int64_t count_ld, const int* __restrict__ count_slot, const float* __restrict__ freq_pen,
    const float* __restrict__ pres_pen, float* __restrict__ ws, int S) {
  __shared__ float red[16];
  __shared__ float redv[16];
  __shared__ int redi[16];
  const int row = blockIdx.y, s = blockIdx.x;
  if (active && !active[row]) return;
  const T* p = logits + (size_t)row * ld;
  const float temp = temperature ? temperature[row] : 1.f;
  const bool greedy = temp <= 0.f;
  const uint64_t step = step_ptr ? (uint64_t)step_ptr[0] : 0;
  const uint64_t ctr0 = step * (uint64_t)((V + 3) / 4);
  const int V8 = (reinterpret_cast<uintptr_t>(p) & 15) == 0 ? (V & ~7) : 0;
  const int slot = (counts && count_slot) ? count_slot[row] : -1;
  Row<T> R;
  R.p = p;
  R.cnt = slot >= 0 ? counts + (size_t)slot * count_ld : nullptr;
  R.freq = R.cnt && freq_pen ? freq_pen[row] : 0.f;
  R.pres = R.cnt && pres_pen ? pres_pen[row] : 0.f;
  R.inv_t = greedy ? 1.f : 1.f / temp;
  const bool noise = !greedy;
  const int chunks = V8 >> 3;
  const int per = (chunks + S - 1) / S;
  const int lo = min(chunks, s * per) * 8, hi = min(chunks, (s + 1) * per) * 8;
  float mx = -INFINITY, se = 0.f;
  ArgMax best;
  best.v = -INFINITY;
  best.i = 0x7fffffff;
  constexpr int PF = 4;
  auto slice = [&](auto noise_c) __attribute__((always_inline)) {
    constexpr bool NOISE = decltype(noise_c)::value;
    for (int base = lo + threadIdx.x * 8; base < hi; base += 256 * 8 * PF) {
      float zz[PF][8];
#pragma unroll
      for (int u = 0; u < PF; ++u) {
        const int i8 = base + u * 256 * 8;
        if (i8 < hi) R.z8(i8, zz[u]);
      }
#pragma unroll
      for (int u = 0; u < PF; ++u) {
        const int i8 = base + u * 256 * 8;
        if (i8 >= hi) break;
        float* z = zz[u];
        float m8 = -INFINITY;
#pragma unroll
        for (int j = 0; j < 8; ++j) m8 = fmaxf(m8, z[j]);
        if (m8 > mx) {
          se *= __expf(mx - m8);
          mx = m8;
        }
        if (mx > -INFINITY) {
#pragma unroll
          for (int j = 0; j < 8; ++j) se += __expf(z[j] - mx);
        }
        u32x4 r0, r1;
        if (NOISE) {
          r0 = Philox::gen(seed, (uint64_t)row, ctr0 + (uint64_t)(i8 >> 2));
          r1 = Philox::gen(seed, (uint64_t)row, ctr0 + (uint64_t)(i8 >> 2) + 1);
        }
        ArgMax c;  // of these eight: the first of the largest
        c.v = -INFINITY;
        c.i = i8;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float key = NOISE ? z[j] + gumbel(j < 4 ? r0[j] : r1[j - 4]) : z[j];
          if (key > c.v) {
            c.v = key;
            c.i = i8 + j;
          }
        }
        best = amax(best, c);
      }
    }
  };
  if (noise) slice(std::true_type{});
  else slice(std::false_type{});
  if (s == S - 1) {  // the entries behind the last whole group of 8 (or the whole row when it is not 16-byte aligned)
    for (int i = V8 + threadIdx.x; i < V; i += 256) {
      const float z = R.z1(i);
      if (z > mx) {
        se *= __expf(mx - z);
        mx = z;
      }
      if (mx > -INFINITY) se += __expf(z - mx);
      ArgMax c;
      c.v = z;
      c.i = i;
      if (noise) c.v += gumbel(Philox::gen(seed, (uint64_t)row, ctr0 + (uint64_t)(i >> 2))[i & 3]);
      best = amax(best, c);
    }
  }
  const float mx_all = block_max(mx, red);
  se = block_sum(mx > -INFINITY ? se * __expf(mx - mx_all) : 0.f, red);
  best = block_argmax(best, redv, redi);
  if (threadIdx.x == 0) {
    float* o = ws + ((size_t)row * S + s) * 4;
    o[0] = mx_all;
    o[1] = se;
    o[2] = best.v;
    o[3] = __int_as_float(best.i);
  }
}

// One wave a row, a lane a slice: a thread a row read its slices one after the other (sampling 1 / 16 / 64 / 320
// rows of 151936 entries, with it, 15.6 / 18.4 / 27.0 / 69.3 -> 10.8 / 13.1 / 21.3 / 66.4 us).
template <typename T>
__global__ __launch_bounds__(64) void sample_combine_kernel(const T* __restrict__ logits, int64_t ld, int V, int B,
                                      const float* __restrict__ temperature, int64_t* __restrict__ step_ptr,
                                      int bump_step, int64_t* __restrict__ out_tok, float* __restrict__ out_logp,
                                      const int* __restrict__ active, int16_t* __restrict__ counts, int64_t count_ld,
                                      const int* __restrict__ count_slot, const float* __restrict__ freq_pen,
                                      const float* __restrict__ pres_pen, const float* __restrict__ ws, int S) {
  const int row = blockIdx.x, lane = threadIdx.x;
  if (row == 0 && lane == 0 && bump_step && step_ptr) step_ptr[0] += 1;  // every reader of the step ran in the previous kernel
  const f32x4 o = lane < S ? *reinterpret_cast<const f32x4*>(ws + ((size_t)row * S + lane) * 4)
                           : (f32x4){-INFINITY, 0.f, -INFINITY, __int_as_float(0x7fffffff)};
  if (active && !active[row]) {
    if (lane != 0) return;
    out_tok[row] = 0;
    if (out_logp) out_logp[row] = 0.f;
    return;
  }
  float mx = o[0];
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) mx = fmaxf(mx, __shfl_xor(mx, d, 64));
  ArgMax best;
  best.v = o[2];
  best.i = __float_as_int(o[3]);
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    ArgMax c;
    c.v = __shfl_xor(best.v, d, 64);
    c.i = __shfl_xor(best.i, d, 64);
    best = amax(best, c);
  }
  const float scale = o[0] > -INFINITY ? __expf(o[0] - mx) : 0.f;
  float se = 0.f;  // in the order of the slices
  for (int s = 0; s < S; ++s)
    se += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(o[1]), s)) *
          __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(scale), s));
  if (lane != 0) return;
  const float temp = temperature ? temperature[row] : 1.f;
  const int slot = (counts && count_slot) ? count_slot[row] : -1;
  Row<T> R;
  R.p = logits + (size_t)row * ld;
  R.cnt = slot >= 0 ? counts + (size_t)slot * count_ld : nullptr;
  R.freq = R.cnt && freq_pen ? freq_pen[row] : 0.f;
  R.pres = R.cnt && pres_pen ? pres_pen[row] : 0.f;
  R.inv_t = temp <= 0.f ? 1.f : 1.f / temp;
  int tok = best.i;
  if (tok < 0 || tok >= V) tok = 0;
  out_tok[row] = tok;
  if (out_logp) out_logp[row] = R.z1(tok) - (mx + __logf(se));
  if (slot >= 0) {
    int16_t* cnt = counts + (size_t)slot * count_ld;
    if (cnt[tok] < 32767) cnt[tok] += 1;
  }
}

// Workspace floats the split path needs for B rows, and the number of slices per row it will use.
extern "C" int areal_sample_splits(int B) {
  if (B >= 1024) return 1;
  const int s = (1024 + B - 1) / B;
  return s > 16 ? 16 : s;
}


extern "C" int areal_sample_unfiltered(const void* logits, int dtype, int B, int V, int64_t ld,
                                       const float* temperature, uint64_t seed, int64_t* step_ptr, int bump_step,
                                       int64_t* out_tok, float* out_logp, const int* active, int16_t* counts,
                                       int64_t count_ld, const int* count_slot, const float* freq_pen,
                                       const float* pres_pen, float* ws, int S, hipStream_t st) {
  if (B == 0) return 0;
  if (S < 1 || S > 64 || !ws) return (int)hipErrorInvalidValue;
  if (counts && (count_ld % 8 != 0 || count_ld < V)) return (int)hipErrorInvalidValue;
  const dim3 grid(S, B);
  if (dtype == 0) {
    hipLaunchKernelGGL(sample_partial_kernel<bf16_t>, grid, dim3(256), 0, st, (const bf16_t*)logits, ld, V,
                       temperature, seed, step_ptr, active, counts, count_ld, count_slot, freq_pen, pres_pen, ws, S);
    hipLaunchKernelGGL(sample_combine_kernel<bf16_t>, dim3(B), dim3(64), 0, st, (const bf16_t*)logits, ld, V, B,
                       temperature, step_ptr, bump_step, out_tok, out_logp, active, counts, count_ld, count_slot,
                       freq_pen, pres_pen, ws, S);
  } else {
    hipLaunchKernelGGL(sample_partial_kernel<float>, grid, dim3(256), 0, st, (const float*)logits, ld, V,
                       temperature, seed, step_ptr, active, counts, count_ld, count_slot, freq_pen, pres_pen, ws, S);
    hipLaunchKernelGGL(sample_combine_kernel<float>, dim3(B), dim3(64), 0, st, (const float*)logits, ld, V, B,
                       temperature, step_ptr, bump_step, out_tok, out_logp, active, counts, count_ld, count_slot,
                       freq_pen, pres_pen, ws, S);
  }
  return (int)hipGetLastError();
}

__global__ void bump_step_kernel(int64_t* step_ptr) {
  if (threadIdx.x == 0 && blockIdx.x == 0) step_ptr[0] += 1;
}

extern "C" int areal_sample(const void* logits, int dtype, int B, int V, int64_t ld,
                            const float* temperature, const int* top_k, const float* top_p,
                            uint64_t seed, int64_t* step_ptr, int bump_step, int64_t* out_tok,
                            float* out_logp, const int* active, int16_t* counts, int64_t count_ld,
                            const int* count_slot, const float* freq_pen, const float* pres_pen,
                            float* ws, int S, hipStream_t st) {
  if (B == 0) return 0;
  if (counts && (count_ld % 8 != 0 || count_ld < V)) return (int)hipErrorInvalidValue;
  if (ws && (S < 1 || S > SLICES || (uintptr_t)ws % 8 != 0)) return (int)hipErrorInvalidValue;
  if (ws) {
    const dim3 grid(S, B), block(SLICE_THREADS);
    if (dtype == 0)
      hipLaunchKernelGGL(sample_slice_kernel<bf16_t>, grid, block, 0, st, (const bf16_t*)logits, ld, V, temperature, top_k, top_p,
                         step_ptr, active, counts, count_ld, count_slot, freq_pen, pres_pen, ws, S);
    else
      hipLaunchKernelGGL(sample_slice_kernel<float>, grid, block, 0, st, (const float*)logits, ld, V, temperature, top_k, top_p,
                         step_ptr, active, counts, count_ld, count_slot, freq_pen, pres_pen, ws, S);
  }
  if (dtype == 0)
    hipLaunchKernelGGL(sample_kernel<bf16_t>, dim3(B), dim3(1024), 0, st, (const bf16_t*)logits, ld, V,
                       temperature, top_k, top_p, seed, step_ptr, out_tok, out_logp, active, counts, count_ld,
                       count_slot, freq_pen, pres_pen, ws, S, bump_step);
  else
    hipLaunchKernelGGL(sample_kernel<float>, dim3(B), dim3(1024), 0, st, (const float*)logits, ld, V,
                       temperature, top_k, top_p, seed, step_ptr, out_tok, out_logp, active, counts, count_ld,
                       count_slot, freq_pen, pres_pen, ws, S, bump_step);
  if (bump_step && step_ptr && !ws)
    hipLaunchKernelGGL(bump_step_kernel, dim3(1), dim3(64), 0, st, step_ptr);
  return (int)hipGetLastError();
}
