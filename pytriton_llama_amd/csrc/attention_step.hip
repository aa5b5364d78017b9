// Attention of a step that brings prompt portions beside decoding requests, in one launch: the workgroups of attention_prefill.hip
// first, behind them those of the decode kernel of attention.hip (bfloat16, head sizes 64 and 128, over the same pages).
//
// Why one launch: a portion's workgroups are bound by what their waves do in a key tile, one of them a compute unit and some units
// without, a decoding request's by the memory that a unit has under way. One after the other each left the
// chip to the other's idle part; here a unit holds two or three workgroups of either kind. Portions take four waves a
// workgroup (one group of them), for a second workgroup to fit beside: eight waves with twice the buffers would keep a unit at head size
// 128 to themselves. The two as branches of a recorded graph overlap as well, but the branch costs about 12 us a layer.
// us, one launch after the other and here (a portion beside 32 rows, 20 of them requests of 130 to 2,900 keys): 24 heads of 128 on 8, 512 rows
// on 512 / 1,536 / 3,072 keys 46.4 / 62.3 / 84.9 -> 39.7 / 45.5 / 76.5, 100 rows on 1,100 55.3 -> 37.7; beside 16 rows, 300 rows on
// 300 keys 21.7 -> 13.0; 32 heads of 64 on 8, 512 rows on 512 / 1,536 29.4 / 38.1 -> 22.4 / 28.0, 1,024 rows 35.6 -> 29.5, 32 rows on
// 1,000 38.1 -> 26.3, beside 64 rows 512 on 512 32.3 -> 24.9, beside 4 of 20 to 300 keys 15.4 -> 10.7. The portions' one group of
// waves is the slower one behind a long prefix, which few or short requests beside it don't make up for at head size 128: 512
// rows on 1,536 / 3,072 keys beside 6 of 20 to 200 keys 38.6 / 61.4 -> 38.3 / 71.4. Hence from eight requests on there, from three
// at 64 (24.4 -> 23.6 on 1,536 keys), and for as many blocks as two groups of waves would take: beyond, one group is
// what they have anyway, and more of their workgroups come before a request's.
#include "attention_decode.h"
#include "attention_prefill.h"
#include "common.h"
#include "device.h"

template <int ND, bool LISTED>
__global__ void __launch_bounds__(256, ND <= 2 ? 3 : 2)
attn_step_kernel(const int32_t* __restrict__ ctx_len, const int32_t* __restrict__ block_table,
                 const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache, const int32_t* __restrict__ q_start,
                 int n_portion_groups, int bt_stride, int n_groups, int Hq, int Hkv, int page_size, int page_shift,
                 const bf16_t* __restrict__ q, long q_stride, bf16_t* __restrict__ out, long out_stride,
                 const int32_t* __restrict__ work_seq, const int32_t* __restrict__ work_qoff, int n_work, int n_seq,
                 int num_splits, int cus, int piece, DecodeParts parts, AttnExtras ex, float scale_log2) {
  constexpr int D = 32 * ND;
  __shared__ __attribute__((aligned(1024))) bf16_t Ks0[PF_BN * D];
  __shared__ __attribute__((aligned(1024))) bf16_t Ks1[PF_BN * D];
  __shared__ __attribute__((aligned(1024))) bf16_t Vs0[PF_BN * D];
  __shared__ __attribute__((aligned(1024))) bf16_t Vs1[PF_BN * D];
  static_assert(decode_region<ND, 2>() <= PF_BN * D * 2, "a wave of a decoding request has one of them");
  const int block = blockIdx.x;
  if (block < n_portion_groups) {
    const int group = block / Hq;                  // (heads fastest, as attention_prefill.hip's grid has them)
    attn_prefill_blocks<ND, ND, 1, bf16_t, false, false, 1, true>(
        Ks0, Ks1, Vs0, Vs1, block - group * Hq, group, n_groups, out, out_stride, q, q_stride, k_cache, v_cache, q_start, ctx_len,
        block_table, bt_stride, work_seq, work_qoff, n_work, Hq, Hkv, 1, page_size, page_shift, ex, scale_log2, 0.f);
  } else {
    attn_decode_part<ND, 2, LISTED, false, false>(
        block - n_portion_groups,
        [&](int w) { return reinterpret_cast<float*>(w == 0 ? Ks0 : w == 1 ? Ks1 : w == 2 ? Vs0 : Vs1); }, ctx_len, block_table,
        k_cache, v_cache, n_seq, Hkv, num_splits, bt_stride, page_size, page_shift, q, q_stride, Hq, cus, piece, out, out_stride,
        q_start, parts, ex, scale_log2, 0.f);
  }
}

// Sequences 0 .. n_seq - 1 bring one token each, the work list (of 64-row blocks, n_groups workgroups a head) names those
// of the others. parts, tickets, most: as for ptl_attention_decode_mfma; page sizes are powers of two from 16 on; no capped
// scores, no kept keys.
extern "C" int ptl_attention_step(void* out, long out_stride, const void* q, long q_stride, const void* k_cache,
                                  const void* v_cache, const int32_t* q_start, const int32_t* ctx_len,
                                  const int32_t* block_table, int bt_stride, const int32_t* work_seq, const int32_t* work_qoff,
                                  int n_work, int n_groups, float* parts, int* tickets, int most, int n_seq, int Hq, int Hkv,
                                  int D, int page_size, int window, int chunk, const float* sink, const float* gate,
                                  long gate_stride, float scale, int num_splits, hipStream_t stream) {
  const AttnExtras ex{window, 0, chunk, sink, gate, gate_stride, 0.f};
  if (n_seq <= 0 || n_work <= 0 || n_groups < 1 || n_groups > n_work || Hq <= 0 || Hkv <= 0 || Hq % Hkv || Hq / Hkv > 16 ||
      Hq > 65535 || (D != 64 && D != 128) || page_size < 16 || (page_size & (page_size - 1)) ||
      (long)Hkv * page_size * D * 2 >= (1L << 32) || q_stride % 8 || out_stride % 4 || num_splits < 1 || num_splits > 1024 ||
      most < num_splits || (most > 1 && (!parts || !tickets)) || !extras_ok(ex))
    return PTL_ERR_ARG;
  const int cus = compute_units(), piece = decode_piece(D, num_splits);
  const bool listed = decode_listed(n_seq);
  const long portions = (long)n_groups * Hq;
  const long decodes = decode_groups(n_seq, Hkv, most, listed, cus);
  if (portions + decodes > 0x7fffffff) return PTL_ERR_ARG;
  const DecodeParts dp{parts, parts ? parts + (long)n_seq * Hq * most * D : nullptr, tickets, most};
  int page_shift = 0;
  while ((1 << page_shift) < page_size) ++page_shift;
#define GO(ND, LISTED)                                                                                                       \
  attn_step_kernel<ND, LISTED><<<(unsigned)(portions + decodes), 256, 0, stream>>>(                                          \
      ctx_len, block_table, (const bf16_t*)k_cache, (const bf16_t*)v_cache, q_start, (int)portions, bt_stride, n_groups, Hq, \
      Hkv, page_size, page_shift, (const bf16_t*)q, q_stride, (bf16_t*)out, out_stride, work_seq, work_qoff, n_work, n_seq,  \
      num_splits, cus, piece, dp, ex, scale * 1.4426950408889634f)
  if (D == 64) {
    if (listed) GO(2, true); else GO(2, false);
  } else {
    if (listed) GO(4, true); else GO(4, false);
  }
#undef GO
  return ptl_launch_status();
}
