// What lies between the attentions of a step of prompts that is launched kernel by kernel (several prompts in a step:
// the steps that are not recorded), one call a layer: what the parts' forward functions launch one by one from Python, in
// their order, with their arguments. Such a step at the 1B shape has 130 kernels, and Python took about 17 us for each, of
// which the launch itself is 5: 2.3 ms for eight prompts of 277 tokens in all, whose kernels take 1.7.
//
// Nothing is decided here: which product goes where is the step's, and the entries that are called (of the
// other libraries, handed over as addresses) check their own arguments; the one that refuses is named in the step.
#include "common.h"

// (in the order of Entry)
struct PtlPromptEntries {
  int (*product)(void*, const void*, const void*, int, int, int, long, long, int, int, long, long, long, int, hipStream_t);
  int (*rope_store)(void*, void*, const void*, long, const int32_t*, const float*, const int32_t*, void*, void*, int, int, int,
                    int, int, int, int, hipStream_t);
  int (*sums)(float*, const void*, const void*, int, int, int, long, int, hipStream_t);
  int (*sum_norm)(void*, const float*, int, void*, const float*, int, int, float, hipStream_t);
  int (*add_norm)(void*, const void*, void*, const float*, int, int, float, int, hipStream_t);
  int (*gate_up)(void*, const void*, const void*, int, int, int, long, int, float, int, hipStream_t);
  int (*act_mul)(void*, const void*, int, int, int, int, hipStream_t);
  int (*qkv)(void*, long, const void*, const void*, int, int, long, const void*, const int32_t*, void*, void*, int, int, int,
             int, int, hipStream_t);
};

enum Entry { PRODUCT, ROPE_STORE, SUMS, SUM_NORM, ADD_NORM, GATE_UP, ACT_MUL, QKV };

// Of the whole step. failed: which Entry a call that returned an error got it from (-1: its own arguments). o_splits, down_splits: slices of K of the tile product, 0: the library's product and the norm by
// itself. gate_up_tile: whether gate and up go through the tile product.
struct PtlPromptStep {
  int T, H, I, Hq, Hkv, D, page_size, act;
  int o_splits, down_splits, gate_up_tile, failed;
  const int32_t *positions, *slots;
  // rows of the step: y (normed) [T, H], residual [T, H], qkv [T, (Hq + 2 Hkv) D], mixed [T, Hq D], a [T, I]; product: the
  // partial sums, or a product [T, H]; gate_up [T, 2 I] (not used where the tile product takes it). qkv, product and
  // gate_up may be one place: none is read any more when the next of them is written.
  void *y, *residual, *qkv, *mixed, *product, *gate_up, *a;
  int qkv_tile;                                  // q | k | v with rotation and cache write in tiles (of qkv only the columns of q are written)
};

struct PtlPromptLayer {
  const void *qkv, *o, *gate_up, *down;
  const float *inv_freq, *post_norm, *next_norm; // next_norm: of the layer behind this one
  void *k_cache, *v_cache;
  float post_eps, next_eps;
  const void* turns;                             // where it says where the cosines and sines of the step's rows lie (qkv_tile)
};

static_assert(sizeof(PtlPromptStep) == 128 && sizeof(PtlPromptLayer) == 88, "as ops/prompt.py lays them out");

// What is behind the attention of ``before`` (null: none) up to the norm in front of ``after``, then what is in
// front of the attention of ``after`` (null: the down projection of ``before`` and the norm are left to the caller).
extern "C" int ptl_prompt_between(const PtlPromptEntries* e, PtlPromptStep* s, const PtlPromptLayer* before,
                                  const PtlPromptLayer* after, hipStream_t st) {
  if (s) s->failed = -1;
  if (!e || !s || s->T <= 0) return PTL_ERR_ARG;
  const int T = s->T, H = s->H, D = s->D, width = (s->Hq + 2 * s->Hkv) * D;
  int rc;
  auto of = [&](Entry which, int code) {
    if (code) s->failed = which;
    return code;
  };
  // x W^T with sum, residual and norm behind it, into y
  auto product_norm = [&](const void* x, const void* w, int K, int splits, const float* norm, float eps) {
    if (splits > 0) {
      float* parts = reinterpret_cast<float*>(s->product);
      const int r = of(SUMS, e->sums(parts, x, w, T, H, K, K, splits, st));
      return r ? r : of(SUM_NORM, e->sum_norm(s->y, parts, splits, s->residual, norm, T, H, eps, st));
    }
    const int r = of(PRODUCT, e->product(s->product, x, w, T, H, K, K, H, PTL_DTYPE_BF16, 1, 0, 0, 0, 0, st));
    return r ? r : of(ADD_NORM, e->add_norm(s->y, s->product, s->residual, norm, T, H, eps, PTL_DTYPE_BF16, st));
  };
  if (before) {
    if ((rc = product_norm(s->mixed, before->o, s->Hq * D, s->o_splits, before->post_norm, before->post_eps))) return rc;
    if (s->gate_up_tile) {
      if ((rc = of(GATE_UP, e->gate_up(s->a, s->y, before->gate_up, T, s->I, H, H, s->act, 0.f, s->act == GLU_SILU, st))))
        return rc;
    } else {
      if ((rc = of(PRODUCT, e->product(s->gate_up, s->y, before->gate_up, T, 2 * s->I, H, H, 2 * s->I, PTL_DTYPE_BF16, 1, 0, 0,
                                       0, 0, st))))
        return rc;
      if ((rc = of(ACT_MUL, e->act_mul(s->a, s->gate_up, T, s->I, s->act, PTL_DTYPE_BF16, st)))) return rc;
    }
    if (after && (rc = product_norm(s->a, before->down, s->I, s->down_splits, before->next_norm, before->next_eps))) return rc;
  }
  if (after && s->qkv_tile) {
    if ((rc = of(QKV, e->qkv(s->qkv, width, s->y, after->qkv, T, H, H, after->turns, s->slots, after->k_cache, after->v_cache,
                             s->Hq, s->Hkv, D, s->page_size, -1, st))))
      return rc;
  } else if (after) {
    if ((rc = of(PRODUCT, e->product(s->qkv, s->y, after->qkv, T, width, H, H, width, PTL_DTYPE_BF16, 1, 0, 0, 0, 0, st))))
      return rc;
    bf16_t* q = reinterpret_cast<bf16_t*>(s->qkv);
    bf16_t *k = q + (size_t)s->Hq * D, *v = k + (size_t)s->Hkv * D;
    if ((rc = of(ROPE_STORE, e->rope_store(q, k, v, width, s->positions, after->inv_freq, s->slots, after->k_cache,
                                           after->v_cache, T, s->Hq, s->Hkv, D, s->page_size, 0, PTL_DTYPE_BF16, st))))
      return rc;
  }
  return PTL_OK;
}
