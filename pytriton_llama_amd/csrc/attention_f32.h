// Attention over a float32 paged cache on the matrix cores, float32 products and
// sums throughout (v_mfma_f32_16x16x4_f32). What the vector kernel of attention.hip takes, for key and
// value sizes that are multiples of 4 up to 128 and 16-byte aligned rows; included by attention.hip.
//
// A workgroup takes a block of 16 query rows and HPW query heads that read one key and value head
// (HPW 2 or 1); its four waves are HPW heads x 4 / HPW parts of the keys. Tiles of BN keys and their
// values come through LDS, two buffers: the next tile is on its way to registers while this one is
// used, its page numbers a tile earlier still. A wave computes S^T = K Q^T, 16 keys x 16 queries at a
// time: lane l (ln = l % 16, lg = l / 16) gets the scores of query ln with keys 4 lg + r, so maxima and
// sums over keys stay in a lane but for two exchanges between lane groups, and the weights are where
// O^T += V^T P^T wants them: the instruction's k = lg of step s is key 4 lg + s in both operands. Four
// steps of a product take a lane's four consecutive floats of a row, read at once: of K and Q along the
// head dimension; of V a lane reads floats 4 ln .. 4 ln + 3 of a group of 64, element t of them going to
// the t-th of four result tiles (whose row i is then value column 4 i + t).
//
// Bound by the matrix cores: 16 keys x 16 queries cost (Dk + Dv) / 4 instructions of 32 clocks against 8 KB
// of LDS reads at head size 64. Rows of keys lie 4 floats apart from a multiple of 64 banks, so that the
// 16 rows of a fragment meet no bank twice; rows of values are read along the row and need no padding.
//
// Measured (one MI355X, us a launch; the vector kernel before in brackets): 700 tokens, 32 heads on 8, head
// size 64: 58 (447); 150 and 333 tokens, 16 heads on one latent head of 128, values of 96: 36 (253);
// 700 tokens, 24 heads of 128 on 8: 146 (897), 16 heads of 16 on 4: 34 (207); 64 rows on 1,500 keys, 8 x 128: 98 (1,451);
// one token behind 333 to 601 keys of four sequences, 32 heads on 8, head size 64, 32 splits planned: 9.3 (24.9).
#pragma once
#include "attention.h"
#include "device.h"
#include "mfma.h"
#include "mfma_f32.h"
#include <type_traits>

#define AF_ROWS 16

// Where a decoded token's keys are cut (see below), of num_splits parts of multiples of AF_DECODE_TILE keys.
#define AF_DECODE_TILE 128
struct SplitArgs {
  float *part_acc, *part_ml;     // [sequence][head][num_splits][Dv] and [2]
  int* tickets;                  // [sequence][kv head][TICKET]: parts that are done, zero before and after the launch
  int num_splits;
};

// DECODE: sequence blockIdx.x brings one token, and the rows of the block are the query heads (up to 16) of kv head
// blockIdx.y; the keys are shared by blockIdx.z workgroups as well, of which the one that is done last merges the parts (a
// second kernel for that took 4.9 us, also where one part has all keys). (HPW 1, maps 1.)
template <int HPW, int NK, int BN, bool DECODE>
__global__ void __launch_bounds__(256)
attn_f32_kernel(float* __restrict__ out, long out_stride, const float* __restrict__ q, long q_stride,
                const float* __restrict__ k_cache, const float* __restrict__ v_cache,
                const int32_t* __restrict__ q_start, const int32_t* __restrict__ ctx_len,
                const int32_t* __restrict__ block_table, int bt_stride, const int32_t* __restrict__ work_seq,
                const int32_t* __restrict__ work_qoff, int Hq, int Hkv, int maps, int Dk, int Dv, int page_size,
                AttnExtras ex, float scale, SplitArgs sp) {
  constexpr int KS = 4 / HPW;                    // parts of the keys
  constexpr int NG = BN / 16 / KS;               // groups of 16 keys of a tile that a wave takes
  constexpr int D = 16 * NK, KLD = D + 4;        // padded sizes; floats between rows of keys in LDS
  constexpr int PIECES = D / 4, PER_PASS = 256 / PIECES, P = BN / PER_PASS;
  static_assert(NG >= 1 && P >= 1, "a tile has 16 keys a part and a row a thread");
  extern __shared__ float lds[];
  float* Ks = lds;                               // [2][BN][KLD]
  float* Vs = lds + 2 * BN * KLD;                // [2][BN][D]
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, ln = lane & 15, lg = lane >> 4;
  const int part = wave / HPW, G = (Hq / maps) / Hkv;
  const int seq = DECODE ? blockIdx.x : work_seq[blockIdx.x], qoff = DECODE ? 0 : work_qoff[blockIdx.x];
  const int qs = q_start[seq], qlen = DECODE ? 1 : q_start[seq + 1] - qs, ctx = ctx_len[seq];
  const int rows = DECODE ? G : min(AF_ROWS, qlen - qoff);
  if (rows <= 0) return;
  // this lane's query: head and row of the batch
  const int head = DECODE ? blockIdx.y * G + min(ln, G - 1) : blockIdx.y * HPW + wave % HPW;
  const int row = qs + (DECODE ? 0 : qoff + ln);
  const int vh = DECODE ? blockIdx.y : (head / maps) / G, kh = DECODE ? vh : vh * maps + head % maps, Hk = Hkv * maps;
  const int32_t* bt = block_table + (size_t)seq * bt_stride;
  const int first_q = ctx - qlen + qoff, qpos = DECODE ? first_q : first_q + ln;
  const int k_end = DECODE ? ctx : min(ctx, first_q + rows), k_lo = first_seen(ex, first_q), row_lo = first_seen(ex, qpos);
  // the walk: the kept first keys left of the window, then the keys from the window's start on
  const int n_kept = min(max(ex.keep_first, 0), k_lo), shift = k_lo - n_kept, n_all = n_kept + (k_end - k_lo);
  int k_first = 0, n_walk = n_all, n_parts = 1;
  if (DECODE) {
    const int per = keys_a_split(n_all, sp.num_splits, AF_DECODE_TILE);
    k_first = blockIdx.z * per;
    n_walk = min(n_all, k_first + per);
    n_parts = max(1, (n_all + per - 1) / per);
    if (blockIdx.z >= n_parts) return;                   // (the first answers for a row without keys)
  }
  const bool row_valid = ln < rows;

  F4 qf[NK];
#pragma unroll
  for (int c = 0; c < NK; ++c)
    qf[c].u = row_valid && 16 * c + 4 * lg < Dk
                  ? load16(q + (size_t)row * q_stride + (size_t)head * Dk + 16 * c + 4 * lg) : zero16();

  const int piece = tid % PIECES, row0 = tid / PIECES;
  int page[P], slot[P];
  uint4 kr[P], vr[P];
  auto pages = [&](int k0) {                     // where the rows of the tile from k0 on lie (page -1: nowhere)
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int kw = k0 + row0 + i * PER_PASS, kp = kw < n_kept ? kw : kw + shift;
      page[i] = kw < n_walk ? bt[kp / page_size] : -1;
      slot[i] = kp % page_size;
    }
  };
  auto fetch = [&]() {
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const bool ok = page[i] >= 0;
      kr[i] = ok && 4 * piece < Dk
                  ? load16(k_cache + (((size_t)page[i] * Hk + kh) * page_size + slot[i]) * Dk + 4 * piece) : zero16();
      vr[i] = ok && 4 * piece < Dv
                  ? load16(v_cache + (((size_t)page[i] * Hkv + vh) * page_size + slot[i]) * Dv + 4 * piece) : zero16();
    }
  };
  auto put = [&](int b) {
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int r = b * BN + row0 + i * PER_PASS;
      *reinterpret_cast<uint4*>(Ks + r * KLD + 4 * piece) = kr[i];
      *reinterpret_cast<uint4*>(Vs + r * D + 4 * piece) = vr[i];
    }
  };
  f32x4_t acc[NK];
#pragma unroll
  for (int t = 0; t < NK; ++t) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;          // l_run: of this lane's keys only

  if (n_walk > k_first) {
    pages(k_first);
    fetch();
    pages(k_first + BN);
    put(0);
  }
  __syncthreads();
  int buf = 0;
  for (int k0 = k_first; k0 < n_walk; k0 += BN, buf ^= 1) {
    const bool more = k0 + BN < n_walk;
    if (more) {
      fetch();
      pages(k0 + 2 * BN);
    }
    f32x4_t s[NG];
    float tmax = -INFINITY;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int base = 16 * (g * KS + part);
      const float* krow = Ks + (buf * BN + base + ln) * KLD + 4 * lg;
      s[g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NK; ++c) {
        F4 kf;
        kf.u = load16(krow + 16 * c);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          s[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf.f[i], qf[c].f[i], s[g], 0, 0, 0);
      }
    }
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int kw = k0 + 16 * (g * KS + part) + 4 * lg + r, kp = kw < n_kept ? kw : kw + shift;
        const bool vis = row_valid && kw < n_walk && kp <= qpos && (kp >= row_lo || kp < ex.keep_first);
        s[g][r] = vis ? cap_score(ex, s[g][r] * scale) : -INFINITY;
        tmax = fmaxf(tmax, s[g][r]);
      }
    tmax = max_with_lane_xor32(max_with_lane_xor16(tmax));
    const float m_new = fmaxf(m_run, tmax);
    const float m_safe = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = expf(m_run - m_safe);
    float psum = 0.f;
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[g][r] = expf(s[g][r] - m_safe);
        psum += s[g][r];
      }
    l_run = l_run * alpha + psum;
    m_run = m_new;
#pragma unroll
    for (int t = 0; t < NK; ++t) acc[t] *= alpha;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const float* vrow = Vs + (buf * BN + 16 * (g * KS + part) + 4 * lg) * D;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (NK >= 4) {
#pragma unroll
          for (int v = 0; v < NK / 4; ++v) {
            F4 vf;
            vf.u = load16(vrow + r * D + 64 * v + 4 * ln);
#pragma unroll
            for (int t = 0; t < 4; ++t)
              acc[4 * v + t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf.f[t], s[g][r], acc[4 * v + t], 0, 0, 0);
          }
        } else {
          const float2 vf = *reinterpret_cast<const float2*>(vrow + r * D + 2 * ln);
          acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf.x, s[g][r], acc[0], 0, 0, 0);
          acc[NK > 1 ? 1 : 0] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf.y, s[g][r], acc[NK > 1 ? 1 : 0], 0, 0, 0);
        }
      }
    }
    if (more) put(buf ^ 1);
    __syncthreads();
  }
  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);

  {                                              // the parts of the keys meet in the first wave of a head
    float* mine = lds + (size_t)wave * (NK * 256 + 128);
    if (part > 0) {
#pragma unroll
      for (int t = 0; t < NK; ++t) *reinterpret_cast<f32x4_t*>(mine + (t * 64 + lane) * 4) = acc[t];
      mine[NK * 256 + lane] = m_run;
      mine[NK * 256 + 64 + lane] = l_run;
    }
    __syncthreads();
    if (part > 0 && !(DECODE && n_parts > 1)) return;
    if (part == 0) {
#pragma unroll
      for (int p = 1; p < KS; ++p) {
        const float* other = lds + (size_t)(wave + p * HPW) * (NK * 256 + 128);
        const float m_o = other[NK * 256 + lane], l_o = other[NK * 256 + 64 + lane];
        const float m_new = fmaxf(m_run, m_o), m_safe = m_new == -INFINITY ? 0.f : m_new;
        const float a = expf(m_run - m_safe), b = expf(m_o - m_safe);
        l_run = l_run * a + l_o * b;
        m_run = m_new;
#pragma unroll
        for (int t = 0; t < NK; ++t)
          acc[t] = acc[t] * a + *reinterpret_cast<const f32x4_t*>(other + (t * 64 + lane) * 4) * b;
      }
    }
  }
  if (DECODE && n_parts > 1) {
    const size_t place = ((size_t)seq * Hq + head) * sp.num_splits + blockIdx.z;
    int* done = reinterpret_cast<int*>(lds);     // (the first wave has left nothing there)
    if (part == 0 && row_valid) {
      if (lg == 0) {
        put_shared(sp.part_ml + place * 2, m_run);
        put_shared(sp.part_ml + place * 2 + 1, l_run);
      }
      float* o = sp.part_acc + place * Dv;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (NK >= 4) {
#pragma unroll
          for (int v = 0; v < NK / 4; ++v) {
            const int d = 64 * v + 16 * lg + 4 * r;
            if (d < Dv) {
#pragma unroll
              for (int t = 0; t < 4; ++t) put_shared(o + d + t, acc[4 * v + t][r]);
            }
          }
        } else {
          const int d = 8 * lg + 2 * r;
          if (d < Dv) { put_shared(o + d, acc[0][r]); put_shared(o + d + 1, acc[NK > 1 ? 1 : 0][r]); }
        }
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // the part has reached memory
    if (tid == 0) *done = last_part(sp.tickets + ((size_t)seq * Hkv + vh) * TICKET, n_parts);
    __syncthreads();
    if (!*done) return;
    // Four columns a thread. The parts lie a long way off: up to eight are asked for at once, in loads of eight bytes (32 rows of 16
    // heads of 96 on one kv head, two parts each: one wave with loads of four bytes, eight parts always, cost a step of eight
    // layers 50 us more than a second kernel).
    auto merge = [&](auto at_once) __attribute__((always_inline)) {
      constexpr int AHEAD = decltype(at_once)::value;
      for (int i = tid; i < G * Dv / 4; i += 256) {
        const int h = 4 * i / Dv, d = 4 * i - h * Dv, hd = vh * G + h;
        const size_t p = ((size_t)seq * Hq + hd) * sp.num_splits;
        const float *pa = sp.part_acc + p * Dv + d, *ml = sp.part_ml + p * 2;
        f32x4_t a = f32x4_t{0.f, 0.f, 0.f, 0.f};
        float mn = ex.sink ? ex.sink[hd] : -INFINITY, den = ex.sink ? 1.f : 0.f;   // (the denominator's term without a key)
        for (int s0 = 0; s0 < n_parts; s0 += AHEAD) {
          float2 lo[AHEAD], hi[AHEAD], ends[AHEAD];
          float m_new = mn;
#pragma unroll
          for (int s = 0; s < AHEAD; ++s) {
            const int at = min(s0 + s, n_parts - 1);
            ends[s] = get_shared2(ml + 2 * at);
            lo[s] = get_shared2(pa + (size_t)at * Dv);
            hi[s] = get_shared2(pa + (size_t)at * Dv + 2);
          }
#pragma unroll
          for (int s = 0; s < AHEAD; ++s) m_new = fmaxf(m_new, ends[s].x);
          const float ms = m_new == -INFINITY ? 0.f : m_new, f0 = expf(mn - ms);
          den *= f0;
          a *= f0;
#pragma unroll
          for (int s = 0; s < AHEAD; ++s) {
            const float f = s0 + s < n_parts ? expf(ends[s].x - ms) : 0.f;
            den = fmaf(ends[s].y, f, den);
            a += f32x4_t{lo[s].x, lo[s].y, hi[s].x, hi[s].y} * f;
          }
          mn = m_new;
        }
        const float inv = den > 0.f ? head_gate(ex, row, hd) / den : 0.f;
        *reinterpret_cast<f32x4_t*>(out + (size_t)row * out_stride + (size_t)hd * Dv + d) = a * inv;
      }
    };
    if (n_parts <= 2) merge(std::integral_constant<int, 2>{});
    else merge(std::integral_constant<int, 8>{});
    return;
  }
  if (!row_valid) return;
  float den = l_run, f = 1.f;
  if (ex.sink) {                                 // one more term of the denominator: exp(sink)
    const float sk = ex.sink[head], mx = fmaxf(m_run, sk);
    f = expf(m_run - mx);
    den = l_run * f + expf(sk - mx);
  }
  const float inv = den > 0.f ? f / den * head_gate(ex, row, head) : 0.f;
  float* o = out + (size_t)row * out_stride + (size_t)head * Dv;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (NK >= 4) {
#pragma unroll
      for (int v = 0; v < NK / 4; ++v) {
        const int d = 64 * v + 16 * lg + 4 * r;
        if (d < Dv)
          *reinterpret_cast<float4*>(o + d) = make_float4(acc[4 * v][r] * inv, acc[4 * v + 1][r] * inv,
                                                          acc[4 * v + 2][r] * inv, acc[4 * v + 3][r] * inv);
      }
    } else {
      const int d = 8 * lg + 2 * r;
      if (d < Dv) *reinterpret_cast<float2*>(o + d) = make_float2(acc[0][r] * inv, acc[NK > 1 ? 1 : 0][r] * inv);
    }
  }
}

template <int HPW, int NK, int BN, bool DECODE, typename... Args>
static int launch_attn_f32(dim3 grid, hipStream_t st, Args... args) {
  constexpr int D = 16 * NK;
  const size_t tiles = (size_t)2 * BN * (2 * D + 4) * sizeof(float);
  const size_t merge = (size_t)4 * (NK * 256 + 128) * sizeof(float);
  const size_t bytes = tiles > merge ? tiles : merge;
  if (bytes > 64 * 1024) {                       // more than a kernel gets unasked
    static LdsAllowance allowance;
    if (!allowance.ask(reinterpret_cast<const void*>(&attn_f32_kernel<HPW, NK, BN, DECODE>), bytes)) return PTL_ERR_ARG;
  }
  attn_f32_kernel<HPW, NK, BN, DECODE><<<grid, 256, bytes, st>>>(args...);
  return ptl_launch_status();
}

static bool attn_f32_fits(const void* out, long out_stride, const void* q, long q_stride, const void* k, const void* v,
                          int Dk, int Dv) {
  return Dk % 4 == 0 && Dv % 4 == 0 && Dk <= 128 && Dv <= 128 && out_stride % 4 == 0 && q_stride % 4 == 0 &&
         (((uintptr_t)out | (uintptr_t)q | (uintptr_t)k | (uintptr_t)v) & 15) == 0;
}

// (arguments as ptl_attention_generic_kv, of attn_f32_fits)
static int attention_f32(float* out, long out_stride, const float* q, long q_stride, const float* k_cache,
                         const float* v_cache, const int32_t* q_start, const int32_t* ctx_len,
                         const int32_t* block_table, int bt_stride, const int32_t* work_seq, const int32_t* work_qoff,
                         int n_work, int Hq, int Hkv, int maps, int Dk, int Dv, int page_size, const AttnExtras& ex,
                         float scale, hipStream_t st) {
  // two heads that share a key head share its tiles; the other waves share the keys. (By the heads alone:
  // how a row's keys are cut, and with it the order of its sums, does not depend on what else is in the step.)
  const int hpw = maps == 1 && Hq / Hkv % 2 == 0 ? 2 : 1;
  const int size = Dk > Dv ? Dk : Dv;
#define GO(HPW, NK, BN)                                                                                            \
  return launch_attn_f32<HPW, NK, BN, false>(dim3(n_work, Hq / HPW), st, out, out_stride, q, q_stride, k_cache, v_cache, \
                                             q_start, ctx_len, block_table, bt_stride, work_seq, work_qoff, Hq, Hkv,    \
                                             maps, Dk, Dv, page_size, ex, scale, SplitArgs{nullptr, nullptr, nullptr, 1})
#define GO_HEADS(NK)             \
  {                              \
    if (hpw == 2) GO(2, NK, 32); \
    GO(1, NK, 64);               \
  }
  if (size <= 32) GO_HEADS(2)
  if (size <= 64) GO_HEADS(4)
  GO_HEADS(8)
#undef GO_HEADS
#undef GO
}

// Where a decoded token takes this kernel (sizes in steps of 16 come here), one map and at most 16 heads a kv head:
// key and value sizes from 32 to 64 always; above 64 from 8, below 32 from 4 heads a kv head on. Against the vector kernel (one
// MI355X, 1 to 40 sequences of 60 to 2,000 keys), us before and with this kernel: sizes 32 to 64 1.25 to 1.67 times as fast
// in the mean of a shape, at worst level but for one head a kv head over 32 kv heads and 2,000 keys (119, 123). Above 64
// the buffers leave room for one workgroup a compute unit (133 KB), and how much of a tile's 16 rows are heads
// decides: 16 on one latent head of 128, 14 sequences of 222 to 1,015 keys 33, 20, 16 of 2,000 40, 19; 16 on 2 x 128 44, 34;
// 24 on 3 x 96 57, 46; but 16 on 4 x 128 46, 58 and 8 on 8 x 128 66, 89. Below 32 half of every tile is padding: 32 on 8 x 16,
// 16 of 2,000 24 to 36 (4 and 8 splits planned), 25 to 23; 32 on 32 x 16, 40 of 2,000 97, 143.
static bool attn_f32_decodes(int Hq, int Hkv, int maps, int Dk, int Dv) {
  const int size = Dk > Dv ? Dk : Dv, heads = Hq / Hkv;
  return maps == 1 && heads <= 16 && Hkv <= 65535 && size <= 128 && heads >= (size > 64 ? 8 : size < 32 ? 4 : 1);
}

// One token a sequence (arguments as ptl_attention_decode_kv, of attn_f32_fits and attn_f32_decodes). Splits without
// keys leave at once.
static int attention_f32_decode(float* out, long out_stride, const float* q, long q_stride, const float* k_cache,
                                const float* v_cache, const int32_t* q_start, const int32_t* ctx_len,
                                const int32_t* block_table, int bt_stride, const SplitArgs& sp, int n_seq, int Hq, int Hkv,
                                int Dk, int Dv, int page_size, const AttnExtras& ex, float scale, hipStream_t st) {
#define GO(NK)                                                                                                    \
  return launch_attn_f32<1, NK, 64, true>(dim3(n_seq, Hkv, sp.num_splits), st, out, out_stride, q, q_stride, k_cache, \
                                          v_cache, q_start, ctx_len, block_table, bt_stride, (const int32_t*)nullptr, \
                                          (const int32_t*)nullptr, Hq, Hkv, 1, Dk, Dv, page_size, ex, scale, sp)
  const int size = Dk > Dv ? Dk : Dv;
  if (size <= 32) GO(2);
  if (size <= 64) GO(4);
  GO(8);
#undef GO
}
