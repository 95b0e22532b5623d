// The layers of a short prefill behind cached context, queued by one call: per layer the split-K qkv product, its row kernel (sum,
// bias, norms, rotation, cache write), attention on the pages, the o product, its row kernel (sum, residual, norm), gate|up with its
// activation, the down product and its row kernel. Host code only: the kernels are those of decode_swiglu.hip, decode_gemm.hip and
// flash_attn_paged.hip through their own entries, and every check is theirs.
//
// What bounded such a prefill is the host: 252 launches of 28 layers took 2250 us to queue from Python, of 2640 in all, where the
// kernels took 1950 (93 tokens behind 811); from here 650, in a few calls that the caller prepares one ahead of the other.
#include <hip/hip_runtime.h>
#include <stdint.h>

extern "C" {
int areal_dtile_slab(const void* X, long xs, const void* W, void* Y, int M, int N, int K, int ct, int mblocks, int ksplit, int stages,
                     int nt, hipStream_t st);
int areal_dswiglu(const void* X, long xs, const void* W, void* Y, long ys, int M, int F, int K, int w, int mblocks, int stages, int nt,
                  int act, hipStream_t st);
int areal_splitk_residual_rmsnorm(const float* slab, int S, const void* bias, const void* res, const void* w, void* res_out, void* y,
                                  int M, int N, float eps, int gemma, hipStream_t st);
int areal_splitk_rope_cache_write(const float* slab, int S, const void* bias, const int* pos, const int64_t* slots, const float* cos_t,
                                  const float* sin_t, void* q_out, void* kcache, void* vcache, int T, int Hq, int Hkv, int D,
                                  int max_pos, int do_rope, const void* q_norm, const void* k_norm, float norm_eps, int fp8,
                                  hipStream_t st);
int areal_flash_fwd_paged(const void* q, const void* kcache, const void* vcache, const int* block_tables, int max_pages, void* o,
                          float* lse, const int* cu_q, const int* cu_k, int B, int max_q, int total_q, int Hq, int Hkv, int D,
                          int64_t q_stride, int64_t o_stride, float softmax_scale, int causal, int fp8, float* part, int splits,
                          hipStream_t st);
}

// One layer's tensors. `next_norm`: the norm behind the layer (null: none, `x` is then the residual stream itself).
struct PrefillLayer {
  const void *qkv, *qkv_bias, *q_norm, *k_norm, *o, *norm2, *gate_up, *down, *next_norm;
  void *kcache, *vcache;
};
struct PrefillPass {
  const PrefillLayer* layers;
  const void* first;  // [T, H] bf16: the first layer's normalised input, kept (or x itself: behind the layers of an earlier call)
  void* x;            // [T, H] bf16: the layers' normalised inputs
  const void* stream;  // [T, H] bf16: the residual stream ahead of the first layer, kept
  void* res[2];       // [T, H] bf16 each: written in turn, res[1] by the last layer
  float* slab;       // the largest of the products' partial sums
  void *q, *attn, *act;
  float* part;       // partial results of the key ranges
  const int* pos;
  const int64_t* slots;
  const float *cos_t, *sin_t;
  const int *block_tables, *cu_q, *cu_k;
  int n_layers, T, H, F, Hq, Hkv, D, max_pos, max_pages, B, max_q, splits;
  int qkv_plan[3], o_plan[3], down_plan[3];  // (32-column tiles, row blocks, splits) of each product
  int gate_cols, gate_blocks, act_kind, fp8, gemma;
  float eps, scale;
};

extern "C" int areal_prefill_layers(const PrefillPass* p, hipStream_t st) {
  const int T = p->T, H = p->H, F = p->F, HD = p->Hq * p->D, N = (p->Hq + 2 * p->Hkv) * p->D;
  const void* in = p->stream;
#define RUN(...)                   \
  do {                             \
    const int rc_ = (__VA_ARGS__); \
    if (rc_ != 0) return rc_;      \
  } while (0)
  auto product = [&](const void* x, const void* w, int n, int k, const int* plan) {
    return areal_dtile_slab(x, k, w, p->slab, T, n, k, plan[0], plan[1], plan[2], 4, 1, st);
  };
  for (int i = 0; i < p->n_layers; ++i) {
    const PrefillLayer& l = p->layers[i];
    RUN(product(i == 0 ? p->first : p->x, l.qkv, N, H, p->qkv_plan));
    RUN(areal_splitk_rope_cache_write(p->slab, p->qkv_plan[2], l.qkv_bias, p->pos, p->slots, p->cos_t, p->sin_t, p->q, l.kcache,
                                      l.vcache, T, p->Hq, p->Hkv, p->D, p->max_pos, 1, l.q_norm, l.k_norm, p->eps, p->fp8, st));
    RUN(areal_flash_fwd_paged(p->q, l.kcache, l.vcache, p->block_tables, p->max_pages, p->attn, nullptr, p->cu_q, p->cu_k, p->B,
                              p->max_q, T, p->Hq, p->Hkv, p->D, HD, HD, p->scale, 1, p->fp8, p->part, p->splits, st));
    RUN(product(p->attn, l.o, H, HD, p->o_plan));
    RUN(areal_splitk_residual_rmsnorm(p->slab, p->o_plan[2], nullptr, in, l.norm2, p->res[0], p->x, T, H, p->eps, p->gemma, st));
    RUN(areal_dswiglu(p->x, H, l.gate_up, p->act, F, T, F, H, p->gate_cols, p->gate_blocks, 4, 1, p->act_kind, st));
    RUN(product(p->act, l.down, H, F, p->down_plan));
    RUN(areal_splitk_residual_rmsnorm(p->slab, p->down_plan[2], nullptr, p->res[0], l.next_norm, p->res[1], l.next_norm ? p->x : p->res[1],
                                      T, H, p->eps, p->gemma, st));
    in = p->res[1];
  }
#undef RUN
  return 0;
}
