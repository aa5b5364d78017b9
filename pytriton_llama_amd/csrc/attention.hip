// Attention over the paged cache for a mixed batch: every query token of a
// sequence attends the keys of that sequence that lie in pages, up to and
// including its own position (its own key was written before the launch).
// A prompt portion and a single decoded token are the same case: q_len rows
// at positions ctx_len - q_len .. ctx_len - 1.
//
// Reference: scores q.k * scale, causal mask, online softmax with running max
// and denominator, float32 accumulators (lite_llama/kernels/flashattentionv2.py:
// 10-61,63-162); query head a reads kv head a / (Hq/Hkv) (:108); the decode
// case is lite_llama/kernels/flashdecoding.py:22-131. The mask of a portion
// with a cached prefix is k_pos <= prefix + q_idx
// (lite_llama/kernels/others/context_flashattention_nopad.py:83-92).
//
// Cache layout: [num_pages, Hkv, page_size, D]; key position p of a sequence is
// in page block_table[seq][p / page_size] at offset p % page_size.
// window > 0 limits a query at position p to keys p-window+1 .. p; pages left
// of every window may be gone (table entry < 0) and are never touched.
// keep_first > 0 (with a window): the keys at positions below keep_first stay visible to every
// later query, at their true positions; their pages are never given back. A kernel walks the
// keys 0 .. min(keep_first, window start) - 1 and then the window, as one list ("walk index":
// index v below n_kept is key v, index v from n_kept on is key v + shift).
// chunk > 0: a query sees the keys of its own chunk only, chunks of so many positions counted from
// position 0; pages of chunks before it may be gone too.
// sink, gate: one more term of a head's denominator, and a factor on its result; softcap: a bound on
// the scores (attention.h).
//
// ptl_attention_generic: vector-FMA kernel, float32 math, storage type T
// (float32 or bfloat16), any page size, any D up to 640 (beyond 256 with more LDS than a
// kernel gets unasked: the launcher asks for it).
#include "attention.h"
#include "attention_decode.h"
#include "attention_f32.h"
#include "common.h"
#include "device.h"
#include "mfma.h"
#include <math.h>

#define BM 16

// NJ: value columns a thread accumulates, 16 apart (16: value sizes up to 256; 40: up to 640).
// Keys of size Dk and values of size Dv need not be alike, and a query head may come in
// ``maps`` forms (several score maps over one set of values): query head j is map j % maps of
// head j / maps, reads key head (kv head) * maps + j % maps and value head (kv head), with
// kv head = (j / maps) / (heads a kv head). TO: the type of the result (T, or float for a
// result that is combined further before it is rounded).
template <typename T, typename TO, int BN, int NJ = 16>
__global__ void __launch_bounds__(256)
attn_generic_kernel(TO* __restrict__ out, long out_stride, const T* __restrict__ q, long q_stride,
                    const T* __restrict__ k_cache, const T* __restrict__ v_cache,
                    const int32_t* __restrict__ q_start, const int32_t* __restrict__ ctx_len,
                    const int32_t* __restrict__ block_table, int bt_stride,
                    const int32_t* __restrict__ work_seq, const int32_t* __restrict__ work_qoff,
                    int Hq, int Hkv, int maps, int Dk, int Dv, int page_size, AttnExtras ex, float scale) {
  extern __shared__ float lds[];
  float* Qs = lds;                   // [BM][Dk]
  float* Ks = Qs + BM * Dk;          // [BN][Dk+1]
  float* Vs = Ks + BN * (Dk + 1);    // [BN][Dv]
  float* Ss = Vs + BN * Dv;          // [BM][BN]

  const int tid = threadIdx.x;
  const int head = blockIdx.y;
  const int seq = work_seq[blockIdx.x];
  const int qoff = work_qoff[blockIdx.x];
  const int qs = q_start[seq];
  const int qlen = q_start[seq + 1] - qs;
  const int ctx = ctx_len[seq];
  const int cached = ctx - qlen;
  const int rows = min(BM, qlen - qoff);
  if (rows <= 0) return;
  const int vh = (head / maps) / ((Hq / maps) / Hkv);      // value head
  const int kh = vh * maps + head % maps;                   // key head (of Hkv * maps)
  const int Hk = Hkv * maps;
  const int32_t* bt = block_table + (size_t)seq * bt_stride;

  for (int i = tid; i < BM * Dk; i += 256) {
    const int m = i / Dk, d = i - m * Dk;
    Qs[i] = m < rows ? to_float<T>(q[(size_t)(qs + qoff + m) * q_stride + head * Dk + d]) : 0.f;
  }

  const int tm = tid >> 4, tc = tid & 15;
  const bool row_valid = tm < rows;
  const int qpos = cached + qoff + tm;
  const int first_q = cached + qoff;
  const int k_end = min(ctx, first_q + rows);
  const int k_lo = first_seen(ex, first_q);
  const int row_lo = first_seen(ex, qpos);
  // the walk: the kept first keys left of the window, then the keys from the window's start on
  const int n_kept = min(max(ex.keep_first, 0), k_lo);
  const int shift = k_lo - n_kept;
  const int n_walk = n_kept + (k_end - k_lo);
  const int nd = (Dv + 15) >> 4;

  float m_run = -INFINITY, l_run = 0.f;
  float acc[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) acc[j] = 0.f;

  for (int k0 = 0; k0 < n_walk; k0 += BN) {
    __syncthreads();
    for (int i = tid; i < BN * Dk; i += 256) {
      const int n = i / Dk, d = i - n * Dk;
      const int kw = k0 + n;
      const int kp = kw < n_kept ? kw : kw + shift;
      float kv = 0.f;
      if (kw < n_walk) {
        const int page = bt[kp / page_size];
        if (page >= 0)
          kv = to_float<T>(k_cache[(((size_t)page * Hk + kh) * page_size + (kp % page_size)) * Dk + d]);
      }
      Ks[n * (Dk + 1) + d] = kv;
    }
    for (int i = tid; i < BN * Dv; i += 256) {
      const int n = i / Dv, d = i - n * Dv;
      const int kw = k0 + n;
      const int kp = kw < n_kept ? kw : kw + shift;
      float vv = 0.f;
      if (kw < n_walk) {
        const int page = bt[kp / page_size];
        if (page >= 0)
          vv = to_float<T>(v_cache[(((size_t)page * Hkv + vh) * page_size + (kp % page_size)) * Dv + d]);
      }
      Vs[i] = vv;
    }
    __syncthreads();

    float s[BN / 16];
    float tmax = -INFINITY;
#pragma unroll
    for (int j = 0; j < BN / 16; ++j) {
      const int n = tc + 16 * j;
      const int kw = k0 + n;
      const int kp = kw < n_kept ? kw : kw + shift;
      const float* qr = Qs + tm * Dk;
      const float* kr = Ks + n * (Dk + 1);
      float dot = 0.f;
      for (int d = 0; d < Dk; ++d) dot = fmaf(qr[d], kr[d], dot);
      const bool vis = row_valid && kw < n_walk && kp <= qpos &&
                       (kp >= row_lo || kp < ex.keep_first);
      s[j] = vis ? cap_score(ex, dot * scale) : -INFINITY;
      tmax = fmaxf(tmax, s[j]);
    }
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) tmax = fmaxf(tmax, __shfl_xor(tmax, o, 64));
    const float m_new = fmaxf(m_run, tmax);
    const float m_safe = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = expf(m_run - m_safe);
    float psum = 0.f;
#pragma unroll
    for (int j = 0; j < BN / 16; ++j) {
      const float p = expf(s[j] - m_safe);
      psum += p;
      Ss[tm * BN + tc + 16 * j] = p;
    }
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) psum += __shfl_xor(psum, o, 64);
    l_run = l_run * alpha + psum;
    m_run = m_new;
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[j] *= alpha;
    __syncthreads();

    const int n_lim = min(BN, n_walk - k0);
    for (int n = 0; n < n_lim; ++n) {
      const float p = Ss[tm * BN + n];
      const float* vr = Vs + n * Dv + tc;
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if (j < nd && tc + 16 * j < Dv) acc[j] = fmaf(p, vr[16 * j], acc[j]);
    }
  }

  if (row_valid) {
    float den = l_run, f = 1.f;
    if (ex.sink) {                         // one more term of the denominator: exp(sink)
      const float sk = ex.sink[head];
      const float mx = fmaxf(m_run, sk);
      f = expf(m_run - mx);
      den = l_run * f + expf(sk - mx);
    }
    const float inv = den > 0.f ? f / den * head_gate(ex, qs + qoff + tm, head) : 0.f;
    TO* o = out + (size_t)(qs + qoff + tm) * out_stride + head * Dv + tc;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      if (j < nd && tc + 16 * j < Dv) o[16 * j] = from_float<TO>(acc[j] * inv);
  }
}

template <typename T, typename TO, int BN, int NJ = 16>
static int launch_generic(void* out, long out_stride, const void* q, long q_stride,
                          const void* k_cache, const void* v_cache, const int32_t* q_start,
                          const int32_t* ctx_len, const int32_t* block_table, int bt_stride,
                          const int32_t* work_seq, const int32_t* work_qoff, int n_work,
                          int Hq, int Hkv, int maps, int Dk, int Dv, int page_size, const AttnExtras& ex,
                          float scale, hipStream_t stream) {
  const size_t lds = (size_t)(BM * Dk + BN * (Dk + 1) + BN * Dv + BM * BN) * sizeof(float);
  if (lds > 64 * 1024) {
    // more dynamic LDS than a kernel may ask for without saying so beforehand (wide heads only)
    static LdsAllowance allowance;
    if (!allowance.ask(reinterpret_cast<const void*>(&attn_generic_kernel<T, TO, BN, NJ>), lds)) return PTL_ERR_ARG;
  }
  dim3 grid(n_work, Hq);
  attn_generic_kernel<T, TO, BN, NJ><<<grid, 256, lds, stream>>>(
      (TO*)out, out_stride, (const T*)q, q_stride, (const T*)k_cache, (const T*)v_cache, q_start,
      ctx_len, block_table, bt_stride, work_seq, work_qoff, Hq, Hkv, maps, Dk, Dv, page_size, ex,
      scale);
  return ptl_launch_status();
}

// The general form. q [T, Hq, Dk] with Hq = heads * maps; k_cache [pages, Hkv * maps, page_size,
// Dk]; v_cache [pages, Hkv, page_size, Dv]; out [T, Hq, Dv] of the caches' type, or float32 when
// out_f32 is set. work_seq / work_qoff list the 16-row query blocks: block i covers rows
// work_qoff[i] .. work_qoff[i]+15 of sequence work_seq[i].
extern "C" int ptl_attention_generic_kv(void* out, long out_stride, int out_f32, const void* q,
                                        long q_stride, const void* k_cache, const void* v_cache,
                                        const int32_t* q_start, const int32_t* ctx_len,
                                        const int32_t* block_table, int bt_stride,
                                        const int32_t* work_seq, const int32_t* work_qoff, int n_work,
                                        int Hq, int Hkv, int maps, int Dk, int Dv, int page_size,
                                        int window, int keep_first, int chunk, const float* sink,
                                        const float* gate, long gate_stride, float softcap, float scale, int dtype,
                                        hipStream_t stream) {
  if (n_work <= 0) return PTL_OK;
  const AttnExtras ex{window, keep_first, chunk, sink, gate, gate_stride, softcap};
  if (Hq <= 0 || Hkv <= 0 || maps <= 0 || Hq % maps || (Hq / maps) % Hkv || Dk <= 0 || Dv <= 0 ||
      Dk > 640 || Dv > 640 || page_size <= 0 || Hq > 65535 || !extras_ok(ex))
    return PTL_ERR_ARG;
#define GO(T, TO, BN, NJ)                                                                         \
  launch_generic<T, TO, BN, NJ>(out, out_stride, q, q_stride, k_cache, v_cache, q_start, ctx_len, \
                                block_table, bt_stride, work_seq, work_qoff, n_work, Hq, Hkv,    \
                                maps, Dk, Dv, page_size, ex, scale, stream)
#define GO_SIZES(T, TO)                                                                           \
  {                                                                                               \
    /* wide heads (a latent cache of 512 + 64, say): 40 columns a thread, 16 keys a turn */       \
    if (Dk > 256 || Dv > 256) return GO(T, TO, 16, 40);                                           \
    return (Dk <= 128 && Dv <= 128) ? GO(T, TO, 32, 16) : GO(T, TO, 16, 16);                      \
  }
  if (dtype == PTL_DTYPE_F32 && attn_f32_fits(out, out_stride, q, q_stride, k_cache, v_cache, Dk, Dv))
    return attention_f32((float*)out, out_stride, (const float*)q, q_stride, (const float*)k_cache,
                         (const float*)v_cache, q_start, ctx_len, block_table, bt_stride, work_seq, work_qoff, n_work,
                         Hq, Hkv, maps, Dk, Dv, page_size, ex, scale, stream);
  if (dtype == PTL_DTYPE_F32) GO_SIZES(float, float)
  if (dtype == PTL_DTYPE_BF16) {
    if (out_f32) GO_SIZES(bf16_t, float)
    GO_SIZES(bf16_t, bf16_t)
  }
#undef GO_SIZES
#undef GO
  return PTL_ERR_ARG;
}

// Keys and values of one size, one score map a head.
extern "C" int ptl_attention_generic(void* out, long out_stride, const void* q, long q_stride,
                                     const void* k_cache, const void* v_cache,
                                     const int32_t* q_start, const int32_t* ctx_len,
                                     const int32_t* block_table, int bt_stride,
                                     const int32_t* work_seq, const int32_t* work_qoff, int n_work,
                                     int Hq, int Hkv, int D, int page_size, int window,
                                     int keep_first, int chunk, const float* sink, const float* gate,
                                     long gate_stride, float softcap, float scale, int dtype, hipStream_t stream) {
  return ptl_attention_generic_kv(out, out_stride, 0, q, q_stride, k_cache, v_cache, q_start, ctx_len,
                                  block_table, bt_stride, work_seq, work_qoff, n_work, Hq, Hkv, 1, D,
                                  D, page_size, window, keep_first, chunk, sink, gate, gate_stride, softcap,
                                  scale, dtype, stream);
}

// ===========================================================================
// ptl_attention_decode: one query token per sequence against its pages, the
// keys split over several workgroups (flash-decoding; the reference's stage 1
// and stage 2 are lite_llama/kernels/flashdecoding.py:22-131 and :171-231:
// every partition emits its accumulator with its running max and denominator,
// the merge weighs them by exp(max_p - max)).
//
// Grid (sequence, kv head x head group, split). A workgroup of four waves
// serves up to GT query heads that share one kv head, so every key and value
// is read once for all of them. A wave reads 64/LPK keys per turn: LPK lanes
// share a key, each lane owns 16 elements of the head dimension of that key
// and of the matching value, for all heads. Every key slot (LPK lanes) keeps
// an online softmax of its own; slots, waves and splits are merged at the end.
// Needs D % 16 == 0. Float32 math throughout.
// ===========================================================================
#define DEC_CHUNK 16

template <typename T> struct Chunk16 { float v[DEC_CHUNK]; };

template <typename T>
__device__ __forceinline__ void load_chunk(const T* __restrict__ p, float* out);

template <>
__device__ __forceinline__ void load_chunk<float>(const float* __restrict__ p, float* out) {
  const float4* p4 = reinterpret_cast<const float4*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float4 x = p4[i];
    out[4 * i] = x.x; out[4 * i + 1] = x.y; out[4 * i + 2] = x.z; out[4 * i + 3] = x.w;
  }
}

template <>
__device__ __forceinline__ void load_chunk<bf16_t>(const bf16_t* __restrict__ p, float* out) {
  const uint4* p4 = reinterpret_cast<const uint4*>(p);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint4 x = p4[i];
    const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      out[8 * i + 2 * j] = __uint_as_float(w[j] << 16);
      out[8 * i + 2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
    }
  }
}

// Keys of size Dk, values of size Dv and ``maps`` score maps a head as in the general form of
// the kernel above: the "kv head" of the grid is a key head (kv head, map); its query heads are
// head * maps + map for the heads of the kv head, its values those of the kv head. LPK lanes cover
// max(Dk, Dv). TO: the type of the result.
template <typename T, typename TO, int GT, int LPK>
__global__ void __launch_bounds__(256)
attn_decode_kernel(TO* __restrict__ out, long out_stride, const T* __restrict__ q, long q_stride,
                   const T* __restrict__ k_cache, const T* __restrict__ v_cache,
                   const int32_t* __restrict__ q_start, const int32_t* __restrict__ ctx_len,
                   const int32_t* __restrict__ block_table, int bt_stride,
                   float* __restrict__ part_acc, float* __restrict__ part_ml,
                   int Hq, int Hkv, int maps, int Dk, int Dv, int page_size, AttnExtras ex, float scale,
                   int num_splits, int groups_per_kv) {
  constexpr int KPW = 64 / LPK;           // keys a wave reads per turn
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int seq = blockIdx.x;
  const int kh = blockIdx.y / groups_per_kv;          // key head: (kv head, map)
  const int hg = blockIdx.y - kh * groups_per_kv;
  const int vh = kh / maps, map = kh - vh * maps;
  const int Hk = Hkv * maps;
  const int split = blockIdx.z;
  const int G = (Hq / maps) / Hkv;
  const int head0 = vh * G + hg * GT;       // first head (of Hq / maps) of this workgroup
  const int nheads = min(GT, G - hg * GT);
  const int row = q_start[seq];
  const int ctx = ctx_len[seq];
  const int k_lo = first_seen(ex, ctx - 1);
  // the walk: the kept first keys left of the window, then the window (indices, not positions)
  const int n_kept = min(max(ex.keep_first, 0), k_lo);
  const int shift = k_lo - n_kept;
  const int span = ctx - shift;
  const int tile = 4 * KPW;
  const int per_split = ((span + num_splits - 1) / num_splits + tile - 1) / tile * tile;
  const int k_begin = split * per_split;
  const int k_end = min(span, k_begin + per_split);
  const int32_t* bt = block_table + (size_t)seq * bt_stride;

  const int c = lane % LPK;                 // which 16 elements of the head this lane owns
  const int ks = lane / LPK;                // key slot within the wave
  const bool active_k = c * DEC_CHUNK < Dk, active_v = c * DEC_CHUNK < Dv;

  float qf[GT][DEC_CHUNK];
#pragma unroll
  for (int h = 0; h < GT; ++h) {
    if (h < nheads && active_k) {
      load_chunk<T>(q + (size_t)row * q_stride + (size_t)((head0 + h) * maps + map) * Dk + c * DEC_CHUNK, qf[h]);
#pragma unroll
      for (int j = 0; j < DEC_CHUNK; ++j) qf[h][j] *= scale;
    } else {
#pragma unroll
      for (int j = 0; j < DEC_CHUNK; ++j) qf[h][j] = 0.f;
    }
  }
  float m[GT], l[GT], acc[GT][DEC_CHUNK];
#pragma unroll
  for (int h = 0; h < GT; ++h) {
    m[h] = -INFINITY; l[h] = 0.f;
#pragma unroll
    for (int j = 0; j < DEC_CHUNK; ++j) acc[h][j] = 0.f;
  }

  for (int kb = k_begin + wave * KPW; kb < k_end; kb += tile) {
    const int kw = kb + ks;
    const bool valid = kw < k_end;
    const int kp = kw < n_kept ? kw : kw + shift;
    float kf[DEC_CHUNK], vf[DEC_CHUNK];
#pragma unroll
    for (int j = 0; j < DEC_CHUNK; ++j) { kf[j] = 0.f; vf[j] = 0.f; }
    if (valid) {
      const int page = bt[kp / page_size];
      const int in_page = kp % page_size;
      if (active_k)
        load_chunk<T>(k_cache + (((size_t)page * Hk + kh) * page_size + in_page) * Dk + c * DEC_CHUNK, kf);
      if (active_v)
        load_chunk<T>(v_cache + (((size_t)page * Hkv + vh) * page_size + in_page) * Dv + c * DEC_CHUNK, vf);
    }
#pragma unroll
    for (int h = 0; h < GT; ++h) {
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < DEC_CHUNK; ++j) s = fmaf(qf[h][j], kf[j], s);
#pragma unroll
      for (int o = 1; o < LPK; o <<= 1) s += __shfl_xor(s, o, 64);
      s = cap_score(ex, s);
      if (valid) {
        if (s > m[h]) {
          const float alpha = expf(m[h] - s);     // exp(-inf) = 0 at the first key
          l[h] *= alpha;
#pragma unroll
          for (int j = 0; j < DEC_CHUNK; ++j) acc[h][j] *= alpha;
          m[h] = s;
        }
        const float p = expf(s - m[h]);
        l[h] += p;
#pragma unroll
        for (int j = 0; j < DEC_CHUNK; ++j) acc[h][j] = fmaf(p, vf[j], acc[h][j]);
      }
    }
  }

  // merge the key slots of the wave
#pragma unroll
  for (int o = LPK; o < 64; o <<= 1) {
#pragma unroll
    for (int h = 0; h < GT; ++h) {
      const float mo = __shfl_xor(m[h], o, 64);
      const float lo = __shfl_xor(l[h], o, 64);
      const float mn = fmaxf(m[h], mo);
      const float ms = mn == -INFINITY ? 0.f : mn;
      const float a = expf(m[h] - ms), b = expf(mo - ms);
      l[h] = l[h] * a + lo * b;
#pragma unroll
      for (int j = 0; j < DEC_CHUNK; ++j)
        acc[h][j] = acc[h][j] * a + __shfl_xor(acc[h][j], o, 64) * b;
      m[h] = mn;
    }
  }

  // merge the four waves through LDS
  extern __shared__ float lds[];
  float* w_acc = lds;                         // [4][GT][Dv]
  float* w_ml = lds + 4 * GT * Dv;            // [4][GT][2]
  if (ks == 0) {
#pragma unroll
    for (int h = 0; h < GT; ++h) {
      if (active_v) {
#pragma unroll
        for (int j = 0; j < DEC_CHUNK; ++j) w_acc[(wave * GT + h) * Dv + c * DEC_CHUNK + j] = acc[h][j];
      }
      if (c == 0) { w_ml[(wave * GT + h) * 2] = m[h]; w_ml[(wave * GT + h) * 2 + 1] = l[h]; }
    }
  }
  __syncthreads();
  for (int i = tid; i < nheads * Dv; i += 256) {
    const int h = i / Dv, d = i - h * Dv;
    float mn = -INFINITY;
#pragma unroll
    for (int w = 0; w < 4; ++w) mn = fmaxf(mn, w_ml[(w * GT + h) * 2]);
    const float ms = mn == -INFINITY ? 0.f : mn;
    float ll = 0.f, a = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = expf(w_ml[(w * GT + h) * 2] - ms);
      ll += w_ml[(w * GT + h) * 2 + 1] * f;
      a += w_acc[(w * GT + h) * Dv + d] * f;
    }
    const int head = (head0 + h) * maps + map;
    if (num_splits == 1) {
      if (ex.sink) {                       // one more term of the denominator: exp(sink)
        const float sk = ex.sink[head];
        const float mx = fmaxf(mn, sk);
        const float f = expf(mn - mx);
        ll = ll * f + expf(sk - mx);
        a *= f;
      }
      out[(size_t)row * out_stride + (size_t)head * Dv + d] =
          from_float<TO>(ll > 0.f ? a / ll * head_gate(ex, row, head) : 0.f);
    } else {
      const size_t pi = ((size_t)seq * Hq + head) * num_splits + split;
      part_acc[pi * Dv + d] = a;
      if (d == 0) { part_ml[pi * 2] = mn; part_ml[pi * 2 + 1] = ll; }
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(64)
attn_decode_merge_kernel(const float* __restrict__ part_acc, const float* __restrict__ part_ml,
                         int Hq, int D, int num_splits, const int32_t* __restrict__ q_start,
                         T* __restrict__ out, long out_stride, AttnExtras ex) {
  // one wave per (sequence, head): lanes take the splits' (max, denominator) side by side,
  // then the head dimension, with the splits' weights in LDS. The partial results come from
  // other compute units' writes, a long way off: the first 16 splits of the lane's first
  // column are asked for before anything is computed, so that one wait covers them and the
  // (max, denominator) pairs.
  constexpr int AHEAD = 16;
  __shared__ float wgt[1024];
  const int seq = blockIdx.x, head = blockIdx.y, lane = threadIdx.x;
  const size_t base = ((size_t)seq * Hq + head) * num_splits;
  const float* pa0 = part_acc + base * D + lane;
  float first[AHEAD];
#pragma unroll
  for (int s = 0; s < AHEAD; ++s) first[s] = (s < num_splits && lane < D) ? pa0[(size_t)s * D] : 0.f;
  const int row = q_start[seq];
  float mn = -INFINITY;
  for (int s = lane; s < num_splits; s += 64) mn = fmaxf(mn, part_ml[(base + s) * 2]);
  mn = wave_max(mn);
  const float sk = ex.sink ? ex.sink[head] : -INFINITY;      // the denominator's term without a key
  mn = fmaxf(mn, sk);
  const float ms = mn == -INFINITY ? 0.f : mn;
  float ll = 0.f;
  for (int s = lane; s < num_splits; s += 64) {
    const float w = expf(part_ml[(base + s) * 2] - ms);
    if (s < 1024) wgt[s] = w;
    ll += part_ml[(base + s) * 2 + 1] * w;
  }
  ll = wave_sum(ll);
  if (ex.sink) ll += expf(sk - ms);
  __syncthreads();
  const float inv = ll > 0.f ? head_gate(ex, row, head) / ll : 0.f;
  for (int d = lane; d < D; d += 64) {
    float a = 0.f;
    const float* pa = part_acc + base * D + d;
    int s = 0;
    if (d == lane) {
#pragma unroll
      for (; s < AHEAD; ++s)
        if (s < num_splits) a = fmaf(first[s], wgt[s], a);
    }
#pragma unroll 8
    for (; s < num_splits; ++s) a = fmaf(pa[(size_t)s * D], wgt[s], a);
    out[(size_t)row * out_stride + (size_t)head * D + d] = from_float<T>(a * inv);
  }
}

template <typename T, typename TO, int LPK>
static int launch_decode(void* out, long out_stride, const void* q, long q_stride,
                         const void* k_cache, const void* v_cache, const int32_t* q_start,
                         const int32_t* ctx_len, const int32_t* block_table, int bt_stride,
                         float* part_acc, float* part_ml, int n_seq, int Hq, int Hkv, int maps, int Dk,
                         int Dv, int page_size, const AttnExtras& ex, float scale, int num_splits,
                         hipStream_t stream) {
  constexpr int GT = 4;
  const int G = (Hq / maps) / Hkv;
  const int groups = (G + GT - 1) / GT;
  dim3 grid(n_seq, Hkv * maps * groups, num_splits);
  const size_t lds = (size_t)(4 * GT * Dv + 4 * GT * 2) * sizeof(float);
  attn_decode_kernel<T, TO, GT, LPK><<<grid, 256, lds, stream>>>(
      (TO*)out, out_stride, (const T*)q, q_stride, (const T*)k_cache, (const T*)v_cache, q_start,
      ctx_len, block_table, bt_stride, part_acc, part_ml, Hq, Hkv, maps, Dk, Dv, page_size, ex,
      scale, num_splits, groups);
  if (hipGetLastError() != hipSuccess) return PTL_ERR_LAUNCH;
  if (num_splits > 1) {
    dim3 mgrid(n_seq, Hq);
    attn_decode_merge_kernel<TO><<<mgrid, 64, 0, stream>>>(part_acc, part_ml, Hq, Dv, num_splits, q_start, (TO*)out,
                                                          out_stride, ex);
  }
  return ptl_launch_status();
}

// Sequences 0..n_seq-1 of the tables each bring one query token (row q_start[s]). q [T, Hq, Dk]
// with Hq = heads * maps, k_cache [pages, Hkv * maps, page_size, Dk], v_cache [pages, Hkv,
// page_size, Dv], out [T, Hq, Dv] of the caches' type or (out_f32) float32.
// part_acc [n_seq, Hq, num_splits, Dv] and part_ml [n_seq, Hq, num_splits, 2] are
// float32 workspaces of the caller (unused when num_splits == 1), and so are, for float32 caches, TICKET * n_seq * Hkv tickets: zeros,
// which they are again after the launch. (Without tickets, or with workspaces that are not 8-byte aligned, which is how the matrix-core
// form reads the parts, the general one takes float32 as well.)
extern "C" int ptl_attention_decode_kv(void* out, long out_stride, int out_f32, const void* q,
                                       long q_stride, const void* k_cache, const void* v_cache,
                                       const int32_t* q_start, const int32_t* ctx_len,
                                       const int32_t* block_table, int bt_stride, float* part_acc,
                                       float* part_ml, int* tickets, int n_seq, int Hq, int Hkv, int maps, int Dk,
                                       int Dv, int page_size, int window, int keep_first, int chunk,
                                       const float* sink, const float* gate, long gate_stride,
                                       float softcap, float scale, int num_splits, int dtype, hipStream_t stream) {
  if (n_seq <= 0) return PTL_OK;
  const AttnExtras ex{window, keep_first, chunk, sink, gate, gate_stride, softcap};
  if (Hq <= 0 || Hkv <= 0 || maps <= 0 || Hq % maps || (Hq / maps) % Hkv || Dk <= 0 || Dk % 16 ||
      Dk > 256 || Dv <= 0 || Dv % 16 || Dv > 256 || page_size <= 0 || num_splits < 1 ||
      num_splits > 1024 || (num_splits > 1 && (!part_acc || !part_ml)) || !extras_ok(ex))
    return PTL_ERR_ARG;
  if (dtype == PTL_DTYPE_F32 && attn_f32_decodes(Hq, Hkv, maps, Dk, Dv) &&
      attn_f32_fits(out, out_stride, q, q_stride, k_cache, v_cache, Dk, Dv) &&
      (num_splits == 1 || (tickets && ((uintptr_t)part_acc | (uintptr_t)part_ml) % 8 == 0)))
    return attention_f32_decode((float*)out, out_stride, (const float*)q, q_stride, (const float*)k_cache,
                                (const float*)v_cache, q_start, ctx_len, block_table, bt_stride,
                                SplitArgs{part_acc, part_ml, tickets, num_splits}, n_seq, Hq, Hkv, Dk, Dv, page_size, ex,
                                scale, stream);
  const int chunks = (Dk > Dv ? Dk : Dv) / 16;
  int lpk = 1;
  while (lpk < chunks) lpk <<= 1;
#define GO(T, TO, L) launch_decode<T, TO, L>(out, out_stride, q, q_stride, k_cache, v_cache, q_start, \
                                             ctx_len, block_table, bt_stride, part_acc, part_ml,    \
                                             n_seq, Hq, Hkv, maps, Dk, Dv, page_size, ex, scale,    \
                                             num_splits, stream)
#define BY_LPK(T, TO)                                                                              \
  switch (lpk) {                                                                                   \
    case 1: return GO(T, TO, 1);                                                                   \
    case 2: return GO(T, TO, 2);                                                                   \
    case 4: return GO(T, TO, 4);                                                                   \
    case 8: return GO(T, TO, 8);                                                                   \
    default: return GO(T, TO, 16);                                                                 \
  }
  if (dtype == PTL_DTYPE_F32) { BY_LPK(float, float) }
  if (dtype == PTL_DTYPE_BF16) {
    if (out_f32) { BY_LPK(bf16_t, float) }
    BY_LPK(bf16_t, bf16_t)
  }
#undef BY_LPK
#undef GO
  return PTL_ERR_ARG;
}

// Keys and values of one size, one score map a head.
extern "C" int ptl_attention_decode(void* out, long out_stride, const void* q, long q_stride,
                                    const void* k_cache, const void* v_cache,
                                    const int32_t* q_start, const int32_t* ctx_len,
                                    const int32_t* block_table, int bt_stride, float* part_acc,
                                    float* part_ml, int* tickets, int n_seq, int Hq, int Hkv, int D, int page_size,
                                    int window, int keep_first, int chunk, const float* sink,
                                    const float* gate, long gate_stride, float softcap, float scale, int num_splits,
                                    int dtype, hipStream_t stream) {
  return ptl_attention_decode_kv(out, out_stride, 0, q, q_stride, k_cache, v_cache, q_start, ctx_len,
                                 block_table, bt_stride, part_acc, part_ml, tickets, n_seq, Hq, Hkv, 1, D, D,
                                 page_size, window, keep_first, chunk, sink, gate, gate_stride, softcap, scale,
                                 num_splits, dtype, stream);
}

// ===========================================================================
// ptl_attention_decode_mfma: the bfloat16 decode case on the matrix cores.
//
// The keys of a (sequence, kv head) pair are cut into equal parts of whole turns, one a workgroup. A pair of one part is
// done with it; the parts of others are merged by the workgroup that is done last, which a counter of the pair says (tickets,
// zero before and after the launch): a second kernel for that costs 4 to 5 us a layer, also where no pair of the
// step has more than one part. Parts and counters are written and read past the XCDs' own L2 (agent scope); nothing waits for
// another workgroup.
//
// What bounds the kernel is the memory a compute unit keeps on its way (about 26 GB/s a unit in all, 17 one workgroup), so its
// time is that of the unit with the most keys, and of the longest part. A pair has num_splits parts of one turn at least, and
// more where they would be longer than ``piece`` keys: the longest sequence of a batch otherwise decides the time of the
// launch. How a pair is cut depends on its own keys and on the launch (num_splits, rows, heads) alone, so a sequence's bits do
// not depend on the others; and so it cannot know whether it is an outlier or one of many equals, for which more parts are more work
// (a part costs 4 to 7 us to begin and to end) and, where some lie above the line and some below, an uneven load.
// Hence the lines (us, 8 kv heads of 64 and of 128): contexts that fill the chip with num_splits parts each lose 5 to 17 % just
// beyond a line, so it lies where such batches are rare, and an outlier is cut as well as a later line allows.
//   one split (two workgroups a unit or about that), 8,192; at 4,096, at the line, not at all: 64 of 3,500 to 5,000 keys 119, 100, 100 and 213,
//   189, 183; of 4,500 110, 105, 101 and 205, 195, 195; 61 to 8,000 98.8, 109, 109 and 192, 186, 187; 7,000 to 10,000 201, 201, 186 and
//   404, 404, 358; 61 to 16,000 184, 186, 209 and 354, 364, 362; one of 8,000 beside 63 of 100 53.1, 93.2, 93.1 and 81, 143, 143, of 16,000
//   54.7, 96.3, 178 and 83, 148, 274. (At 2,048 64 of 2,062, a batch behind prompts of that length, took 54.5 for 49.0, 100 for 92.7.)
//   two and three splits, 2,048 up to 64; at 2,048 and not at all: 32 of 130 to 8,000 51.9, 54.7, of 8,000 93.2, 91.6, of 6,200 78.3, 72.5;
//   one of 8,000 beside 31 of 100 30.4, 37.2. Above 64 1,024; at 2,048, at the line, not at all: 20 of 130 to 2,900 beside 12 empty rows
//   40.5, 32.4, 40.8; one of 3,000 beside 31 of 100 37.7, 28.8, 37.7, of 8,000 47, 47, 80; 32 of 2,000 51.0, 50.7, 51.3, of 2,100 54.5, 58.9,
//   54.0, of 4,000 93.3, 96.3, 93.9, of 8,000 176, 176, 176; 32 of 130 to 4,300 60, 66, 60, to 8,000 108, 110, 102.
//   four (16 requests), 3,072 up to 64 and 4,096 above; at 2,048, 3,072, 4,096, not at all: 16 of 8,300 58.9, 54.4, 52.4, 52.5 and 112, 103,
//   103, 98.9; of 12,300 81.8, 81.5, 77.1, 77.3 and 153, 157, 141, 141; of 16,400 99.4, 98.7, 108, 99.7 and 186, 182, 200, 184; 130 to
//   16,000 54.0, 53.6, 56.2, 56.4 and 111, 105, 101, 96.8; one of 16,000 beside 15 of 100 30.4, 37.4, 52.4, 52.4 and 48.7, 59.9, 82.6, 83.1,
//   of 32,000 beside 15 of 2,000 59, 59, 59, 100 and 94, 94, 94, 160.
//   more (up to 12 requests or so), not at all: a part is short beside the launch. At 2,048 and not at all: 8 of 16,400 56.2, 54.1 and 109, 98.1;
//   of 20,000 69.9, 63.1 and 135, 115; of 32,800 101, 95.1 and 196, 183; 130 to 32,000 76.1, 70.6 and 148, 134; one of 32,000 beside 7 of
//   100 68.5, 71.3 and 136, 135.
// And no pair has more parts than a launch of DECODE_MOST_GROUPS workgroups a unit has room for: the grid is made for the
// longest context that the block table can hold, and workgroups without keys take their place in the queue. 64 of 300 keys, 8 kv heads of
// 64, with a table of 131,072 tokens 19.3 -> 12.0, of 128 29.9 -> 18.7, 256 of 300 55 -> 31 and 96 -> 61, 32 of 100 to 500 15.3 -> 12.3
// and 24.4 -> 18.1: as with a table of 4,096, and with a grid without those workgroups.
// Where the contexts of 9 to 64 sequences differ by more than a quarter (each workgroup finds that out from ctx_len, a recorded step
// does not know it) the parts of all pairs are one list, the longest first, every second turn of the units from the other
// end: a unit's second workgroup is short where its first is long. Equal ones keep the grid's order (64 of 1,400, 8 x 64, 36.1
// against 38.0 in the list).
// Measured (one MI355X, us; with the parts merged by a second kernel and without the list in brackets): one of 45 keys, 8 x 64, 4.8 (6.7);
// one of 2,048 7.7 (8.7); 8 of 2,048 11.9 (12.7), of 300 7.0 (8.4); 16 of 2,000 18.1 (18.8); 64 of 61 to 2,610 40.1 (41.2), of 2,062 49.0
// (50.6), 8 x 128 66.6 (68.0) and 92.7 (96.6); 20 of 130 to 2,900 beside 12 empty rows 20.3 (23.0), 8 x 128 32.4 (44.1); 32 of 2,000, 8 x
// 128, 50.7 (52.5); 48 of 300 to 3,000 35.9 (39.0), 73.1 (72.3). Eight waves a workgroup instead of four: 64 of 1,400, 8 x 64, 36 -> 40. A
// persistent grid that walks the list costs the start of every part again: 64 of 1,400 in two parts 42.7, one workgroup a part 41.6.
//
// A wave takes UNR tiles of 16 keys per turn and all query heads of a kv head at once (up to 16 of them
// are the N side of the MFMA tiles, so grouped heads cost nothing extra):
//   S^T[key, head] = K[key, :] . Q[head, :]         v_mfma_f32_16x16x32_bf16,
//                                                   A = 16-byte loads of key rows
//   O^T[d, head]  += V^T[d, key] . P^T[key, head]   v_mfma_f32_16x16x16_bf16,
//                                                   B = P^T as it leaves the
//                                                   first product, A = V^T
// The value tiles go through a region of LDS that belongs to the wave: written as
// they lie in the cache (rows of D, 16-byte stores), read back transposed with
// ds_read_b64_tr_b16 (in a group of 16 lanes, lane s points at
// V[4 g + s/4][16 t + 4 (s%4)] and lane l receives V[4 g + 0..3][16 t + l]).
// Nothing in the loop over keys waits for another wave. The keys and values of the next turn
// are on their way from global memory while this turn is computed, and the page
// numbers of the turn after that are read one turn earlier still.
// The softmax state of a head (running max, denominator) lives in the lanes of
// that head's column; the waves are merged at the end of a part. Needs D % 32 == 0, D <= 128, Hq/Hkv <= 16, a page size
// that is a power of two, pages (of all kv heads) below 4 GiB.
// ===========================================================================
template <int NDT, int UNR, bool LISTED, bool KEPT, bool CAP>
__global__ void __launch_bounds__(256, NDT <= 2 ? 3 : 2)
attn_decode_mfma_kernel(const int32_t* __restrict__ ctx_len, const int32_t* __restrict__ block_table,
                        const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache, int n_seq, int Hkv,
                        int num_splits, int bt_stride, int page_size, int page_shift, const bf16_t* __restrict__ q, long q_stride,
                        int Hq, int cus, int piece, bf16_t* __restrict__ out, long out_stride,
                        const int32_t* __restrict__ q_start, DecodeParts parts, AttnExtras ex, float scale_log2, float cap_in) {
  extern __shared__ float lds[];
  attn_decode_part<NDT, UNR, LISTED, KEPT, CAP>(
      blockIdx.x, [](int w) { return lds + w * (decode_region<NDT, UNR>() / 4); }, ctx_len, block_table, k_cache, v_cache, n_seq,
      Hkv, num_splits, bt_stride, page_size, page_shift, q, q_stride, Hq, cus, piece, out, out_stride, q_start, parts, ex,
      scale_log2, cap_in);
}

template <int NDT, int UNR, bool LISTED>
static int launch_decode_mfma(void* out, long out_stride, const void* q, long q_stride,
                              const void* k_cache, const void* v_cache, const int32_t* q_start,
                              const int32_t* ctx_len, const int32_t* block_table, int bt_stride,
                              float* parts, int* tickets, int n_seq, int Hq, int Hkv, int page_size, const AttnExtras& ex,
                              float scale, int num_splits, int most, int piece, hipStream_t stream) {
  constexpr int D = 32 * NDT, WAVES = 4;
  const int cus = compute_units();
  const long groups = decode_groups(n_seq, Hkv, most, LISTED, cus);
  if (groups > 0x7fffffff) return PTL_ERR_ARG;
  const DecodeParts dp{parts, parts ? parts + (long)n_seq * Hq * most * D : nullptr, tickets, most};
  int page_shift = 0;
  while ((1 << page_shift) < page_size) ++page_shift;
  const size_t lds = (size_t)WAVES * decode_region<NDT, UNR>();
  const bool kept = ex.window > 0 && ex.keep_first > 0, cap = ex.softcap > 0.f;
  const float log2e = 1.4426950408889634f;
  const float scale_log2 = (cap ? ex.softcap : scale) * log2e, cap_in = cap ? 2.0f * log2e * scale / ex.softcap : 0.f;
#define GO(KEPT, CAP)                                                                                              \
  attn_decode_mfma_kernel<NDT, UNR, LISTED, KEPT, CAP><<<(unsigned)groups, 64 * WAVES, lds, stream>>>(             \
      ctx_len, block_table, (const bf16_t*)k_cache, (const bf16_t*)v_cache, n_seq, Hkv, num_splits, bt_stride, page_size, \
      page_shift, (const bf16_t*)q, q_stride, Hq, cus, piece, (bf16_t*)out, out_stride, q_start, dp, ex, scale_log2, cap_in)
  if (kept) {
    if (cap) GO(true, true); else GO(true, false);
  } else {
    if (cap) GO(false, true); else GO(false, false);
  }
#undef GO
  return ptl_launch_status();
}

// The most parts a pair of at most ``keys`` keys has, of n_seq * Hkv pairs. Where they are more than one, ptl_attention_decode_mfma
// wants n_seq * Hq * parts * (D + 2) floats of workspace and TICKET * n_seq * Hkv tickets. piece: as there; the caller's own is
// not limited by what the launch has room for.
extern "C" int ptl_attention_decode_mfma_parts(int D, int num_splits, long keys, long pairs, int piece) {
  if (D <= 0 || num_splits < 1 || keys <= 0 || pairs <= 0 || piece < 0) return 1;
  if (piece > 0) return max(num_splits, (int)min((keys + piece - 1) / piece, (long)DECODE_MOST_PARTS));
  return decode_most(D, num_splits, keys, pairs, compute_units());
}

// parts: floats of workspace for ``most`` parts a pair (ptl_attention_decode_mfma_parts for at least the keys of the longest
// sequence); tickets: zeros, which they are again after the launch. unroll: 16-key tiles a wave takes per turn, 1 or 2 (0:
// the kernel's choice). piece: keys beyond which a part is cut again (0: the kernel's choice).
extern "C" int ptl_attention_decode_mfma(void* out, long out_stride, const void* q, long q_stride,
                                         const void* k_cache, const void* v_cache,
                                         const int32_t* q_start, const int32_t* ctx_len,
                                         const int32_t* block_table, int bt_stride, float* parts, int* tickets, int most,
                                         int n_seq, int Hq, int Hkv, int D,
                                         int page_size, int window, int keep_first, int chunk,
                                         const float* sink, const float* gate, long gate_stride,
                                         float softcap, float scale, int num_splits, int unroll, int piece,
                                         hipStream_t stream) {
  if (n_seq <= 0) return PTL_OK;
  const AttnExtras ex{window, keep_first, chunk, sink, gate, gate_stride, softcap};
  if (Hq <= 0 || Hkv <= 0 || Hq % Hkv || Hq / Hkv > 16 || D <= 0 || D % 32 || D > 128 ||
      page_size <= 0 || (page_size & (page_size - 1)) || Hq > 65535 ||
      (long)Hkv * page_size * D * 2 >= (1L << 32) || q_stride % 8 || num_splits < 1 ||
      num_splits > 1024 || most < num_splits || (most > 1 && (!parts || !tickets)) || unroll < 0 || unroll > 2 || piece < 0 ||
      !extras_ok(ex))
    return PTL_ERR_ARG;
  if (unroll == 0) unroll = 2;
  if (piece == 0) piece = decode_piece(D, num_splits);
#define GO(N, U)                                                                                                \
  (decode_listed(n_seq)                                                                                              \
       ? launch_decode_mfma<N, U, true>(out, out_stride, q, q_stride, k_cache, v_cache, q_start, ctx_len,       \
                                        block_table, bt_stride, parts, tickets, n_seq, Hq, Hkv, page_size, ex, scale, \
                                        num_splits, most, piece, stream)                                        \
       : launch_decode_mfma<N, U, false>(out, out_stride, q, q_stride, k_cache, v_cache, q_start, ctx_len,      \
                                         block_table, bt_stride, parts, tickets, n_seq, Hq, Hkv, page_size, ex, scale, \
                                         num_splits, most, piece, stream))
  if (unroll == 1) {
    switch (D / 32) {
      case 1: return GO(1, 1);
      case 2: return GO(2, 1);
      case 3: return GO(3, 1);
      default: return GO(4, 1);
    }
  }
  switch (D / 32) {
    case 1: return GO(1, 2);
    case 2: return GO(2, 2);
    case 3: return GO(3, 2);
    default: return GO(4, 2);
  }
#undef GO
}
