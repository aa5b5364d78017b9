// Decode attention over the paged cache on the matrix cores: what a workgroup does, for the kernels of attention.hip (which has the
// reasons and the figures) and attention_step.hip.
#pragma once
#include "attention.h"
#include "common.h"
#include "device.h"
#include "mfma.h"

__device__ __forceinline__ void wave_lds_fence() {
  // orders this wave's LDS writes and reads for the compiler; the LDS itself runs a wave's
  // instructions in order
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

#define DECODE_LIST_SEQS 64        // sequences of a listed launch (one a lane)
#define DECODE_MOST_PARTS 16       // parts that ``piece`` cuts a pair into at most
#define DECODE_MOST_GROUPS 4       // ... as long as the launch has no more workgroups a compute unit than that

// What parts of a pair the workgroups leave for the one that merges them.
struct DecodeParts {
  float *acc, *ml;                 // [sequence][head][most][D] results, [..][2] their maximum (of scores times log2 e) and denominator
  int* tickets;                    // [sequence][kv head][TICKET]: parts that are done
  int most;                        // parts a pair has room for
};

// Bytes of LDS of a wave (attn_decode_part's region): its value tiles, then its sums (and a word for all).
template <int NDT, int UNR> constexpr int decode_region() {
  const int values = UNR * 16 * (32 * NDT + 16) * 2, sums = 16 * (32 * NDT + 2) * 4 + 16;
  return values > sums ? values : sums;
}

// What workgroup ``block`` of four waves does. region(w): LDS of wave w, 16-byte aligned. LISTED: a list of parts (attention.hip),
// cus: the compute units, the grid a multiple of them; else a grid of workgroups (sequence, kv head, split), the sequences fastest.
// KEPT: a window that keeps the sequence's first keys (keep_first > 0). CAP: scores are capped; then
// scale_log2 is softcap * log2 e and cap_in takes a raw score to tanh_exp2's argument.
template <int NDT, int UNR, bool LISTED, bool KEPT, bool CAP, typename Region>
__device__ __forceinline__ void
attn_decode_part(int block, Region region, const int32_t* __restrict__ ctx_len, const int32_t* __restrict__ block_table,
                        const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache, int n_seq, int Hkv,
                        int num_splits, int bt_stride, int page_size, int page_shift, const bf16_t* __restrict__ q, long q_stride,
                        int Hq, int cus, int piece, bf16_t* __restrict__ out, long out_stride,
                        const int32_t* __restrict__ q_start, DecodeParts parts, AttnExtras ex, float scale_log2, float cap_in) {
  constexpr int D = 32 * NDT;
  constexpr int NT = 2 * NDT;             // 16-wide tiles of the head dimension
  constexpr int WAVES = 4;
  constexpr int UNIT = 16 * UNR;          // keys of a wave's turn
  constexpr int TILE = UNIT * WAVES;      // ... of the workgroup's
  constexpr int VS = D + 16;              // row stride of a value tile in LDS, in elements
  constexpr int CPR = D / 8;              // 16-byte chunks per row
  constexpr int VCH = 16 * CPR / 64;      // chunks of a tile per lane
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ln = lane & 15, lg = lane >> 4;
  const int G = Hq / Hkv;
  const int page_mask = page_size - 1;
  const uint32_t page_bytes = (uint32_t)Hkv * page_size * D * 2;
  bf16_t* vl = reinterpret_cast<bf16_t*>(region(wave));
  // this lane's chunks of a value tile: row vrow[i], elements vcol[i] .. +7
  int vrow[VCH], vcol[VCH];
#pragma unroll
  for (int i = 0; i < VCH; ++i) {
    const int c = lane + 64 * i;
    vrow[i] = c / CPR;
    vcol[i] = (c - vrow[i] * CPR) * 8;
  }
  int seq = block % n_seq, kvh = block / n_seq % Hkv, split = block / (n_seq * Hkv), per, n_parts;
  if (LISTED) {
    // lane s has sequence s: the keys of its parts, and how many of them a pair has
    const int c = lane < n_seq ? ctx_len[lane] : 0, keys = c > 0 ? walk_of(ex, c) : 0;
    const int lane_per = keys_a_split(keys, min(max(num_splits, (keys + piece - 1) / piece), parts.most), TILE);   // (below too)
    const int lane_parts = lane < n_seq ? max(1, (keys + lane_per - 1) / lane_per) : 0;
    const unsigned long long some = __ballot(keys > 0);
    const int one = some ? __builtin_amdgcn_readlane(keys, __ffsll(some) - 1) : 0;
    if (__any(keys > 0 && abs(keys - one) > one / 4)) {
      const int turn = block / cus, unit = block - turn * cus, at = turn * cus + (turn % 2 ? cus - 1 - unit : unit);
      const int group = at / (8 * Hkv), in_group = at - group * 8 * Hkv, u = 8 * group + in_group % 8;
      int all = lane_parts;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) all += __shfl_xor(all, o, 64);
      if (u >= all) return;
      // the longest parts first: every wave counts a quarter of the sequences that come before the lane's
      const int packed = (keys > 0 ? min(lane_per, 1 << 24) : 0) << 6 | (63 - lane);
      int start = 0;
      for (int s = __builtin_amdgcn_readfirstlane(wave); s < n_seq; s += WAVES)
        start += __builtin_amdgcn_readlane(packed, s) > packed ? __builtin_amdgcn_readlane(lane_parts, s) : 0;
      reinterpret_cast<int*>(region(wave))[lane] = start;
      __syncthreads();
      start = 0;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) start += reinterpret_cast<const int*>(region(w))[lane];
      __syncthreads();
      seq = __ffsll((unsigned long long)__ballot(u >= start && u < start + lane_parts)) - 1;
      kvh = in_group / 8;
      split = u - __builtin_amdgcn_readlane(start, seq);
    }
    per = __builtin_amdgcn_readlane(lane_per, seq);
    n_parts = __builtin_amdgcn_readlane(lane_parts, seq);
    if (split >= n_parts) return;
  }
  const int head0 = kvh * G;
  const int row = q_start[seq];
  const int ctx = ctx_len[seq];
  const int k_lo = first_seen(ex, ctx - 1);
  // the walk: the kept first keys left of the window, then the window; k_begin, k_end and the
  // keys of a turn are indices of the walk, key_at gives the position
  const int n_kept = KEPT ? min(max(ex.keep_first, 0), k_lo) : 0;
  const int shift = k_lo - n_kept;
  const int span = ctx - shift;
  if (!LISTED) {
    per = keys_a_split(span, min(max(num_splits, (span + piece - 1) / piece), parts.most), TILE);
    n_parts = max(1, (span + per - 1) / per);
    if (split >= n_parts) return;
  }
  const int k_begin = split * per;
  const int k_end = min(span, k_begin + per);
  const int turns = (k_end - k_begin + TILE - 1) / TILE;
  auto key_at = [&](int kw) { return (KEPT && kw < n_kept) ? kw : kw + shift; };
  const int32_t* bt = block_table + (size_t)seq * bt_stride;
  const char* k_head = reinterpret_cast<const char*>(k_cache) + (size_t)kvh * page_size * D * 2;
  const char* v_head = reinterpret_cast<const char*>(v_cache) + (size_t)kvh * page_size * D * 2;

  Frag8 qf[NDT];
#pragma unroll
  for (int kk = 0; kk < NDT; ++kk) {
    qf[kk].u = make_uint4(0, 0, 0, 0);
    if (ln < G)
      qf[kk].u = *reinterpret_cast<const uint4*>(q + (size_t)row * q_stride +
                                                 (size_t)(head0 + ln) * D + 32 * kk + 8 * lg);
  }
  f32x4_t o[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) o[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_part = 0.f;

  int pk[UNR], pv[UNR][VCH];            // pages of the key row and of the value chunks' rows
  uint4 vg[UNR][VCH];                   // values on their way to LDS
  auto first_key = [&](int turn) { return k_begin + turn * TILE + 16 * UNR * wave; };
  auto load_pages = [&](int turn) {
    const int kc = first_key(turn);
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      const int kp = kc + 16 * u + ln;
      pk[u] = (turn < turns && kp < k_end) ? bt[key_at(kp) >> page_shift] : -1;
#pragma unroll
      for (int i = 0; i < VCH; ++i) {
        const int vp = kc + 16 * u + vrow[i];
        pv[u][i] = (turn < turns && vp < k_end) ? bt[key_at(vp) >> page_shift] : -1;
      }
    }
  };
  auto issue_loads = [&](int turn, Frag8 (&kf)[UNR][NDT]) {
    const int kc = first_key(turn);
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      const int kp = key_at(kc + 16 * u + ln);
      const char* kr = k_head + (size_t)(uint32_t)max(pk[u], 0) * page_bytes +
                       (uint32_t)(((kp & page_mask) * D + 8 * lg) * 2);
#pragma unroll
      for (int kk = 0; kk < NDT; ++kk)
        kf[u][kk].u = pk[u] >= 0 ? load_once(kr + 64 * kk) : make_uint4(0, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < VCH; ++i) {
        const int vp = key_at(kc + 16 * u + vrow[i]);
        vg[u][i] = make_uint4(0, 0, 0, 0);              // rows past the end read as zeros
        if (pv[u][i] >= 0)
          vg[u][i] = load_once(v_head + (size_t)(uint32_t)pv[u][i] * page_bytes +
                               (uint32_t)(((vp & page_mask) * D + vcol[i]) * 2));
      }
    }
  };
  // one turn: the values that arrived go to LDS, the next turn's loads are issued, this
  // turn's keys (in kf) and values (in LDS) are used
  auto step = [&](int turn, Frag8 (&kf)[UNR][NDT], Frag8 (&kf_next)[UNR][NDT]) {
    wave_lds_fence();                                   // the last turn's reads are done
#pragma unroll
    for (int u = 0; u < UNR; ++u)
#pragma unroll
      for (int i = 0; i < VCH; ++i)
        *reinterpret_cast<uint4*>(vl + (u * 16 + vrow[i]) * VS + vcol[i]) = vg[u][i];
    wave_lds_fence();
    if (turn + 1 < turns) {
      issue_loads(turn + 1, kf_next);
      load_pages(turn + 2);
    }
    const int kc = first_key(turn);
    if (kc >= k_end) return;                            // wave-uniform: nothing of this turn is ours
    f32x4_t st[UNR];
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      st[u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < NDT; ++kk)
        st[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[u][kk].v, qf[kk].v, st[u], 0, 0, 0);
    }
    float tmax = -INFINITY;
#pragma unroll
    for (int u = 0; u < UNR; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float sc = (CAP ? tanh_exp2(st[u][i] * cap_in) : st[u][i]) * scale_log2;
        sc = (kc + 16 * u + 4 * lg + i < k_end) ? sc : -INFINITY;
        st[u][i] = sc;
        tmax = fmaxf(tmax, sc);
      }
    tmax = max_with_lane_xor16(tmax);
    tmax = max_with_lane_xor32(tmax);
    if (tmax > m_run) {                                 // (finite: key kc is in range)
      const float alpha = __builtin_amdgcn_exp2f(m_run - tmax);
      m_run = tmax;
      l_part *= alpha;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        o[t][0] *= alpha; o[t][1] *= alpha; o[t][2] *= alpha; o[t][3] *= alpha;
      }
    }
    s16x4_t pb[UNR];
#pragma unroll
    for (int u = 0; u < UNR; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p = __builtin_amdgcn_exp2f(st[u][i] - m_run);
        l_part += p;
        pb[u][i] = (short)float_to_bf16(p);
      }
    const bf16_t* vp = vl + (4 * lg + (ln >> 2)) * VS + 4 * (ln & 3);
#pragma unroll
    for (int u = 0; u < UNR; ++u)
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const s16x4_t vf = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4_t*)(vp + u * 16 * VS + 16 * t));
        o[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(vf, pb[u], o[t], 0, 0, 0);
      }
  };

  Frag8 kfa[UNR][NDT], kfb[UNR][NDT];
  load_pages(0);
  issue_loads(0, kfa);
  load_pages(1);
  for (int turn = 0; turn < turns; turn += 2) {
    step(turn, kfa, kfb);
    if (turn + 1 < turns) step(turn + 1, kfb, kfa);
  }
  float l = l_part + __shfl_xor(l_part, 16, 64);
  l += __shfl_xor(l, 32, 64);

  // column d of the h-th head's result: the weighted sum a of values and the denominator ll to the maximum mn
  auto write = [&](int h, int d, float mn, float ll, float a) {
    const int head = head0 + h;
    if (ex.sink) {                         // one more term of the denominator: exp(sink)
      const float sk = ex.sink[head] * 1.4426950408889634f;
      const float mx = fmaxf(mn, sk);
      const float f = __builtin_amdgcn_exp2f(mn - mx);
      ll = ll * f + __builtin_amdgcn_exp2f(sk - mx);
      a *= f;
    }
    // (by the inverse: where a score is a NaN or an infinity, a and ll are NaNs, and so is the result)
    out[(size_t)row * out_stride + (size_t)head * D + d] = float_to_bf16(a * (ll > 0.f ? head_gate(ex, row, head) / ll : 0.f));
  };

  // merge the waves: [head][D] accumulators and [head][2] (max, denominator) take the place of
  // a wave's value tiles, which it has left by now
  __syncthreads();
  if (ln < G) {
    float* const mine = region(wave);
#pragma unroll
    for (int t = 0; t < NT; ++t)
      *reinterpret_cast<f32x4_t*>(mine + ln * D + 16 * t + 4 * lg) = o[t];
    if (lg == 0) { mine[16 * D + ln * 2] = m_run; mine[16 * D + ln * 2 + 1] = l; }
  }
  __syncthreads();
  for (int i = tid; i < G * D; i += 64 * WAVES) {
    const int h = i / D, d = i - h * D;
    float mn = -INFINITY;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) mn = fmaxf(mn, region(w)[16 * D + h * 2]);
    const float ms = mn == -INFINITY ? 0.f : mn;
    float ll = 0.f, a = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float* const part = region(w);
      const float f = __builtin_amdgcn_exp2f(part[16 * D + h * 2] - ms);
      ll += part[16 * D + h * 2 + 1] * f;
      a += part[h * D + d] * f;
    }
    if (n_parts == 1) {
      write(h, d, mn, ll, a);
    } else {
      const size_t p = ((size_t)seq * Hq + head0 + h) * parts.most + split;
      put_shared(parts.acc + p * D + d, a);
      if (d == 0) { put_shared(parts.ml + p * 2, mn); put_shared(parts.ml + p * 2 + 1, ll); }
    }
  }
  if (n_parts > 1) {
    int* done = reinterpret_cast<int*>(region(0) + 16 * (D + 2));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // this wave's part of the part has reached memory
    __syncthreads();
    if (tid == 0) *done = last_part(parts.tickets + ((size_t)seq * Hkv + kvh) * TICKET, n_parts);
    __syncthreads();
    if (*done) {
      // (the parts lie a long way off: eight of them are asked for at once)
      constexpr int AHEAD = 8;
      for (int i = tid; i < G * D; i += 64 * WAVES) {
        const int h = i / D, d = i - h * D;
        const size_t p = ((size_t)seq * Hq + head0 + h) * parts.most;
        const float *acc = parts.acc + p * D + d, *ml = parts.ml + p * 2;
        float mn = -INFINITY, ll = 0.f, a = 0.f;
        for (int s0 = 0; s0 < n_parts; s0 += AHEAD) {
          float av[AHEAD], mv[AHEAD], lv[AHEAD];
#pragma unroll
          for (int s = 0; s < AHEAD; ++s) {
            const int at = min(s0 + s, n_parts - 1);
            mv[s] = get_shared(ml + 2 * at);
            lv[s] = get_shared(ml + 2 * at + 1);
            av[s] = get_shared(acc + (size_t)at * D);
          }
          float m_new = mn;
#pragma unroll
          for (int s = 0; s < AHEAD; ++s) m_new = fmaxf(m_new, mv[s]);
          const float ms = m_new == -INFINITY ? 0.f : m_new, f0 = __builtin_amdgcn_exp2f(mn - ms);
          ll *= f0;
          a *= f0;
#pragma unroll
          for (int s = 0; s < AHEAD; ++s) {
            const float f = s0 + s < n_parts ? __builtin_amdgcn_exp2f(mv[s] - ms) : 0.f;
            ll = fmaf(lv[s], f, ll);
            a = fmaf(av[s], f, a);
          }
          mn = m_new;
        }
        write(h, d, mn, ll, a);
      }
    }
  }
}

// Whether the parts of all pairs are one list.
static bool decode_listed(int n_seq) { return n_seq > 8 && n_seq <= DECODE_LIST_SEQS; }
// The keys beyond which a part is cut again, and the most parts that a pair of at most ``keys`` keys then has (figures in
// attention.hip).
static int decode_piece(int D, int num_splits) {
  if (num_splits > 4) return 1 << 30;
  if (num_splits == 4) return D > 64 ? 4096 : 3072;
  return num_splits == 1 ? 8192 : D > 64 ? 1024 : 2048;
}
static int decode_most(int D, int num_splits, long keys, long pairs, int cus) {
  const int piece = decode_piece(D, num_splits);
  const long cut = min((keys + piece - 1) / piece, (long)DECODE_MOST_PARTS);
  return max(num_splits, (int)min(cut, (long)DECODE_MOST_GROUPS * cus / pairs));
}
// Workgroups of a launch with room for ``most`` parts a pair.
static long decode_groups(int n_seq, int Hkv, int most, bool listed, int cus) {
  if (!listed) return (long)n_seq * Hkv * most;
  return ((long)(n_seq * most + 7) / 8 * 8 * Hkv + cus - 1) / cus * cus;   // (whole turns of the units)
}
