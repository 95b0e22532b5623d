// Launch plans that depend on the number of tokens of a pass and are searched ahead of its first launch: a serving engine's prefills
// seldom repeat a length, and the device waits for the search. Costs are doubles in the order of operations of the Python forms
// (ops/decode_gemm.py, ops/attention.py), so that both choose the same plan.
#pragma once
#include <algorithm>
#include <cstdint>
#include <stdexcept>
#include <tuple>

namespace areal {

constexpr int64_t kPlanCus = 256;

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// A product of M rows, N columns, K deep into partial sums: (32-column tiles a workgroup, row blocks, splits). K >= 64.
inline std::tuple<int64_t, int64_t, int64_t> slab_plan(int64_t M, int64_t N, int64_t K) {
  if (M < 1 || N < 1 || K < 64) throw std::invalid_argument("slab_plan: no rows, no columns or less than 64 deep");
  constexpr int64_t kMost = 24;
  const int64_t steps = K / 64, deep = std::max<int64_t>(1, std::min(kMost, K / 192));
  int64_t per[kMost + 1];  // steps of a split; 0: one of them would have none
  for (int64_t ksplit = 1; ksplit <= deep; ++ksplit) {
    per[ksplit] = ceil_div(steps, ksplit);
    if (per[ksplit] * (ksplit - 1) >= steps) per[ksplit] = 0;
  }
  double best = 0;
  std::tuple<int64_t, int64_t, int64_t> plan{0, 0, 0};
  for (int64_t mblocks = ceil_div(M, 256); mblocks <= ceil_div(M, 32); ++mblocks) {
    const int64_t rt = ceil_div(ceil_div(M, mblocks), 32);
    if (mblocks > 1 && (mblocks - 1) * rt * 32 >= M) continue;  // a row block of no rows
    for (int64_t ct = 1; ct <= 5; ++ct) {
      const int64_t tiles = ceil_div(N, 32 * ct) * mblocks;
      const double step = (double)(46 * (rt + ct)) + 5.6 * (double)rt * (double)ct + 46.0;
      const int64_t rounds = ceil_div(tiles, kPlanCus);  // (of one where there are splits)
      for (int64_t ksplit = 1; ksplit <= deep && (ksplit == 1 || ksplit * tiles <= kPlanCus); ++ksplit) {
        if (per[ksplit] == 0) continue;
        const double cost = (double)(rounds * per[ksplit]) * step + (double)(450 * ksplit * M * N) * 4e-6;
        if (std::get<0>(plan) == 0 || cost < best) {
          best = cost;
          plan = {ct, mblocks, ksplit};
        }
      }
    }
  }
  return plan;
}

// Ranges of keys of a paged prefill of `tiles` (query tile, head) pairs, `rows` (query, head) rows and max_k keys.
inline int64_t key_ranges(int64_t tiles, int64_t rows, int64_t max_k, int64_t workgroups, int64_t keys) {
  if (tiles < 1 || workgroups < 0 || keys < 1) throw std::invalid_argument("key_ranges: no tiles or no keys a range");
  const int64_t walk = ceil_div(max_k, 64);
  const int64_t most = std::max<int64_t>(1, std::min({workgroups / tiles, max_k / keys, (int64_t)32}));
  int64_t plan = 1;
  double best = 0;
  for (int64_t splits = 1; splits <= most; ++splits) {
    const int64_t groups = tiles * splits;
    const double cost = (double)ceil_div(walk, splits) * (groups <= 256 ? 2.1 : 2.7) * std::max(1.0, (double)groups / 512.0) +
                        (splits > 1 ? 4.0 + 3.5e-4 * (double)rows * (double)splits : 0.0);
    if (splits == 1 || cost < best) {
      best = cost;
      plan = splits;
    }
  }
  return plan;
}

}  // namespace areal
