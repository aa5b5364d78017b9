// Attention of prompt portions over the paged cache on the matrix cores (bfloat16).
// The cache layout, the meaning of the arguments and the reference formulas are those of
// attention.hip.
#include "attention_prefill.h"
#include "common.h"
#include "device.h"
#include "mfma.h"
#include <math.h>
#include <type_traits>

// ===========================================================================
// ptl_attention_prefill_mfma: bfloat16 prompt portions on the matrix cores.
//
// A workgroup of four waves (or of eight, which share the keys) takes 64 or 128 query rows of one head (16 or 32 per
// wave) and walks the sequence's keys in tiles of 64. Key and value tiles go
// through LDS as they lie in the cache (rows of D), in two buffers: while tile t
// is used, tile t+1 is on its way from global memory straight into the other
// buffer (global_load_lds_dwordx4, no register in between; its page numbers were
// read one tile earlier still), so a tile costs one barrier. Both products are
// computed transposed so that the scores leave the first MFMA in the register
// layout the second one wants, without a shuffle:
//   S^T[key, query] = K[key, :] . Q[query, :]      (A = K tile, B = Q^T)
//   O^T[d, query]  += V^T[d, key] . P^T[key, query] (A = V^T tile, B = P^T)
// with v_mfma_f32_16x16x32_bf16: a lane holds 8 consecutive k-values of row
// (lane % 16), k-group (lane / 16); the result tile holds rows 4*(lane/16)+i,
// column lane % 16. The V^T fragments come from the row-major value tile through
// ds_read_b64_tr_b16: in a group of 16 lanes, lane s gives the address of four
// consecutive elements E[s][0..3], and lane l receives E[4i + l/4][l%4], i = 0..3;
// with lane s pointing at V[key0 + s/4][d0 + 4*(s%4)], lane l gets
// V[key0 + 0..3][d0 + l]. Softmax is the online one of
// lite_llama/kernels/flashattentionv2.py:10-61 in base 2 (scale * log2 e folded
// into the scores, exp2), float32 max / denominator / accumulator; P is rounded
// to bfloat16 for the second product as there (:55). The running maximum is a
// stabiliser, not a result: it follows the scores only when they pass it by more
// than 8 (in the exponent's units), so that what is kept is rescaled rarely.
// Needs D % 32 == 0, D <= 128, a page size that is a power of two.
//
// Keys of size DK and values of size DV need not be alike (both multiples of 32 up to 128), and
// a head may come in several score maps over one set of values, as in the general form of the
// vector kernel (attention.hip): query head j is map j % maps of head j / maps and reads key
// head (kv head) * maps + j % maps and the values of its kv head. The result is bfloat16, or
// float32 for one that is combined further before it is rounded.
// ===========================================================================

template <int NDK, int NDV, int RT, typename TO, bool KEPT, bool CAP, int SIDES, bool PAGED>
__global__ void __launch_bounds__(256 * SIDES, SIDES == 1 && (NDK + NDV) <= 4 ? 3 : 2)
attn_prefill_mfma_kernel(TO* __restrict__ out, long out_stride, const bf16_t* __restrict__ q,
                         long q_stride, const bf16_t* __restrict__ k_cache,
                         const bf16_t* __restrict__ v_cache, const int32_t* __restrict__ q_start,
                         const int32_t* __restrict__ ctx_len, const int32_t* __restrict__ block_table,
                         int bt_stride, const int32_t* __restrict__ work_seq,
                         const int32_t* __restrict__ work_qoff, int n_work, int Hq, int Hkv, int maps,
                         int page_size, int page_shift, AttnExtras ex, float scale_log2, float cap_in) {
  __shared__ __attribute__((aligned(1024))) bf16_t Ks0[SIDES * PF_BN * 32 * NDK];
  __shared__ __attribute__((aligned(1024))) bf16_t Ks1[SIDES * PF_BN * 32 * NDK];
  __shared__ __attribute__((aligned(1024))) bf16_t Vs0[SIDES * PF_BN * 32 * NDV];
  __shared__ __attribute__((aligned(1024))) bf16_t Vs1[SIDES * PF_BN * 32 * NDV];
  attn_prefill_blocks<NDK, NDV, RT, TO, KEPT, CAP, SIDES, PAGED>(
      Ks0, Ks1, Vs0, Vs1, blockIdx.x, blockIdx.y, gridDim.y, out, out_stride, q, q_stride, k_cache, v_cache, q_start, ctx_len,
      block_table, bt_stride, work_seq, work_qoff, n_work, Hq, Hkv, maps, page_size, page_shift, ex, scale_log2, cap_in);
}

template <int NDK, int NDV, int RT, typename TO, int SIDES>
static int launch_prefill_mfma(void* out, long out_stride, const void* q, long q_stride,
                               const void* k_cache, const void* v_cache, const int32_t* q_start,
                               const int32_t* ctx_len, const int32_t* block_table, int bt_stride,
                               const int32_t* work_seq, const int32_t* work_qoff, int n_work,
                               int n_groups, int Hq, int Hkv, int maps, int page_size, const AttnExtras& ex,
                               float scale, hipStream_t stream) {
  dim3 grid(Hq, n_groups < 65535 ? n_groups : 65535);
  int page_shift = -1;
  for (int sh = 0; sh < 31; ++sh)
    if ((1 << sh) == page_size) page_shift = sh;
  const bool kept = ex.window > 0 && ex.keep_first > 0, cap = ex.softcap > 0.f;
  if (kept && cap) return PTL_ERR_ARG;
  const float log2e = 1.4426950408889634f;
  const float scale_log2 = (cap ? ex.softcap : scale) * log2e, cap_in = cap ? 2.0f * log2e * scale / ex.softcap : 0.f;
  constexpr bool SIZES = NDK != 3 && NDV != 3;
#define GO(KEPT, CAP, PAGED)                                                                                \
  attn_prefill_mfma_kernel<NDK, NDV, RT, TO, KEPT, CAP, SIDES, PAGED><<<grid, 256 * SIDES, 0, stream>>>(    \
      (TO*)out, out_stride, (const bf16_t*)q, q_stride, (const bf16_t*)k_cache, (const bf16_t*)v_cache,     \
      q_start, ctx_len, block_table, bt_stride, work_seq, work_qoff, n_work, Hq, Hkv, maps, page_size,      \
      page_shift, ex, scale_log2, cap_in)
  if (kept) GO(true, false, false);
  else if (cap) GO(false, true, false);
  else if (SIZES && page_size >= 16) GO(false, false, SIZES);
  else GO(false, false, false);
#undef GO
  return ptl_launch_status();
}

// Keys and values of one size, one score map a head, bfloat16 result: the sizes every model
// with ordinary heads brings.
template <int RT, int SIDES>
static int prefill_same_size(int nd, void* out, long out_stride, const void* q, long q_stride,
                             const void* k_cache, const void* v_cache, const int32_t* q_start,
                             const int32_t* ctx_len, const int32_t* block_table, int bt_stride,
                             const int32_t* work_seq, const int32_t* work_qoff, int n_work, int n_groups,
                             int Hq, int Hkv, int page_size, const AttnExtras& ex, float scale,
                             hipStream_t stream) {
#define GO(N) launch_prefill_mfma<N, N, RT, bf16_t, SIDES>(out, out_stride, q, q_stride, k_cache, v_cache, q_start, \
                                                    ctx_len, block_table, bt_stride, work_seq, work_qoff,  \
                                                    n_work, n_groups, Hq, Hkv, 1, page_size, ex, scale,  \
                                                    stream)
  switch (nd) {
    case 1: return GO(1);
    case 2: return GO(2);
    case 3: return GO(3);
    default: return GO(4);
  }
#undef GO
}

// work_seq / work_qoff list query blocks of ``block_rows`` rows (64 or 128), the longest first;
// n_groups workgroups a head share them (1 <= n_groups <= n_work). longest: rows of the longest portion, or the
// most that a recorded step can bring (0: not known). bfloat16 only; q rows must be 16-byte aligned and output rows 8-byte (q_stride % 8, out_stride % 4); the
// page size is a power of two and a page of all kv heads is smaller than 4 GiB.
extern "C" int ptl_attention_prefill_mfma(void* out, long out_stride, const void* q, long q_stride,
                                          const void* k_cache, const void* v_cache,
                                          const int32_t* q_start, const int32_t* ctx_len,
                                          const int32_t* block_table, int bt_stride,
                                          const int32_t* work_seq, const int32_t* work_qoff,
                                          int n_work, int n_groups, int block_rows, int longest, int Hq,
                                          int Hkv, int D,
                                          int page_size, int window, int keep_first, int chunk,
                                          const float* sink, const float* gate, long gate_stride,
                                          float softcap, float scale, hipStream_t stream) {
  if (n_work <= 0) return PTL_OK;
  const AttnExtras ex{window, keep_first, chunk, sink, gate, gate_stride, softcap};
  if (Hq <= 0 || Hkv <= 0 || Hq % Hkv || D % 32 || D <= 0 || D > 128 || page_size <= 0 ||
      (page_size & (page_size - 1)) || (long)Hkv * page_size * D * 2 >= (1L << 32) ||
      Hq > 65535 || n_groups < 1 || n_groups > n_work || q_stride % 8 || out_stride % 4 ||
      (block_rows != 64 && block_rows != 128) || !extras_ok(ex))
    return PTL_ERR_ARG;
  // Two sides where there are few workgroups a compute unit and portions are long enough to have long
  // chains of key tiles by themselves. A block's time is that of its
  // chain of key tiles, and a compute unit with one workgroup of four waves has one wave a SIMD, which
  // nothing covers: eight waves on two chains of half the length hold the unit as well as a second
  // workgroup would, and there is none. Beyond that a unit holds two workgroups of four waves (the
  // buffers of two sides leave no room for a second one), and the chains overlap without this.
  // 24 heads of 128, 512 rows: on 1,536 keys 40.7 -> 29.5 us, on 3,072 76.5 -> 52.5, a prompt of 512
  // 17.4 -> 14.1, of 300 12.1 -> 11.3; 32 heads of 64, 300 rows 8.9 -> 8.0. Below 256 keys the larger workgroup
  // costs 0.2 to 0.8 us (64 rows on 64 keys 6.3 -> 7.1, 128 on 128 7.9 -> 8.6, 200 on 200 level), which every short
  // prompt would pay in every layer; a short portion behind a long prefix gains (64 rows on 320 keys 12.1 ->
  // 11.3, on 1,088 29.9 -> 22.8). How many keys a recorded step will have is not known at its launch: callers give
  // the rows of what is most likely a prompt of its own, and 0 where a prefix is as likely.
  // Up to two workgroups a unit: at head sizes up to 64 two of eight waves fit as well, so two sides win for lists of more than
  // 256 rows (longest not known) or with a portion of 512; above, a unit holds one at a time, and they win for a
  // prompt by itself only, whose workgroups are of all lengths (us with one side and two; 32 heads of 64: 700 rows 13.9 / 11.7,
  // 1,024 18.4 / 15.7, 700 on 3,072 keys 48.5 / 40.9, 1,024 on 4,096 64.5 / 53.5, twice 512 11.5 / 11.1, but three times 260 8.7 /
  // 9.5; 16 heads of 128: 1,531 rows 40.7 / 30.8, 2,048 53.0 / 45.6; 24 of 128: 700 rows 21.4 / 18.2, 1,024 29.0 / 25.2, but
  // 700 on 3,072 keys 78 / 91 and 300 + 200 + 257 + 100 12.6 / 15.6; 32 of 128: twice 512 17.8 / 21.1). Three workgroups a unit are
  // level at head size 64 (1,531 rows of 32 heads 25.9 / 26.4) and lose above (42.1 / 48.0).
  const long groups = (long)n_groups * Hq, units = compute_units();
  const bool both = groups <= units ||
                    (groups <= 2 * units && (D <= 64 ? (longest <= 0 ? n_groups > 4 : longest >= 512)
                                                     : longest > 0 && longest > 64L * (n_work - 2)));
  if (block_rows == 64 && (longest <= 0 || longest > 256) && both)
    return prefill_same_size<1, 2>(D / 32, out, out_stride, q, q_stride, k_cache, v_cache, q_start, ctx_len,
                                   block_table, bt_stride, work_seq, work_qoff, n_work, n_groups, Hq, Hkv,
                                   page_size, ex, scale, stream);
  if (block_rows == 64)
    return prefill_same_size<1, 1>(D / 32, out, out_stride, q, q_stride, k_cache, v_cache, q_start, ctx_len,
                                block_table, bt_stride, work_seq, work_qoff, n_work, n_groups, Hq, Hkv,
                                page_size, ex, scale, stream);
  return prefill_same_size<2, 1>(D / 32, out, out_stride, q, q_stride, k_cache, v_cache, q_start, ctx_len,
                              block_table, bt_stride, work_seq, work_qoff, n_work, n_groups, Hq, Hkv,
                              page_size, ex, scale, stream);
}

// The general form: q [T, Hq, Dk] with Hq = heads * maps, k_cache [pages, Hkv * maps, page_size,
// Dk], v_cache [pages, Hkv, page_size, Dv], out [T, Hq, Dv] bfloat16 or (out_f32) float32; Dk and
// Dv multiples of 32 up to 128. 64-row blocks; longest: as above.
extern "C" int ptl_attention_prefill_mfma_kv(void* out, long out_stride, int out_f32, const void* q,
                                             long q_stride, const void* k_cache, const void* v_cache,
                                             const int32_t* q_start, const int32_t* ctx_len,
                                             const int32_t* block_table, int bt_stride,
                                             const int32_t* work_seq, const int32_t* work_qoff,
                                             int n_work, int n_groups, int longest, int Hq, int Hkv, int maps, int Dk,
                                             int Dv, int page_size, int window, int keep_first, int chunk,
                                             const float* sink, const float* gate, long gate_stride,
                                             float softcap, float scale, hipStream_t stream) {
  if (n_work <= 0) return PTL_OK;
  const AttnExtras ex{window, keep_first, chunk, sink, gate, gate_stride, softcap};
  if (Hq <= 0 || Hkv <= 0 || maps <= 0 || Hq % maps || (Hq / maps) % Hkv || Dk % 32 || Dk <= 0 ||
      Dk > 128 || Dv % 32 || Dv <= 0 || Dv > 128 || page_size <= 0 || (page_size & (page_size - 1)) ||
      (long)Hkv * maps * page_size * Dk * 2 >= (1L << 32) || (long)Hkv * page_size * Dv * 2 >= (1L << 32) ||
      Hq > 65535 || n_groups < 1 || n_groups > n_work || q_stride % 8 || out_stride % 4 || !extras_ok(ex))
    return PTL_ERR_ARG;
  if (Dk == Dv && maps == 1 && !out_f32)         // (one group of waves or two)
    return ptl_attention_prefill_mfma(out, out_stride, q, q_stride, k_cache, v_cache, q_start, ctx_len, block_table, bt_stride,
                                      work_seq, work_qoff, n_work, n_groups, 64, longest, Hq, Hkv, Dk, page_size, window,
                                      keep_first, chunk, sink, gate, gate_stride, softcap, scale, stream);
#define GO(NK, NV, TO)                                                                                  \
  launch_prefill_mfma<NK, NV, 1, TO, 1>(out, out_stride, q, q_stride, k_cache, v_cache, q_start, ctx_len, \
                                     block_table, bt_stride, work_seq, work_qoff, n_work, n_groups, Hq, \
                                     Hkv, maps, page_size, ex, scale, stream)
#define BY_V(NK, TO)                   \
  switch (Dv / 32) {                   \
    case 1: return GO(NK, 1, TO);      \
    case 2: return GO(NK, 2, TO);      \
    case 3: return GO(NK, 3, TO);      \
    default: return GO(NK, 4, TO);     \
  }
#define BY_K(TO)                       \
  switch (Dk / 32) {                   \
    case 1: BY_V(1, TO)                \
    case 2: BY_V(2, TO)                \
    case 3: BY_V(3, TO)                \
    default: BY_V(4, TO)               \
  }
  if (out_f32) { BY_K(float) }
  BY_K(bf16_t)
#undef BY_K
#undef BY_V
#undef GO
}
