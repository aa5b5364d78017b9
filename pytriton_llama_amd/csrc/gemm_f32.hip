// y = x W^T in float32 on the matrix cores: row-major x [M, K] (row stride ldx) and W [N, K]; both are split into three
// bfloat16 parts, whose products are exact, and the sums are float32 (split_f32.h).
//
// All kernels need K % 4 == 0 and 16-byte aligned rows of x and W; everything else stays with the
// vector-FMA kernel.
//
// One order of sums. The bits of a result do not depend on the other rows of x, nor on how many there are, so
// that a request's float32 results are the same alone and in a batch: all kernels add the products of a result
// in an order that K alone fixes. The columns are cut into spans of span_width(K) (at most 16), a span into blocks of 32
// columns. A block's sum starts from zero and takes six matrix instructions; a span's starts from zero and takes its
// blocks' one after the other; the spans' sums are added in order. Which wave, workgroup or lane computes a span is free.
// (Measured against the float32 matrix instructions, which add four columns at a time, with sums of even and odd blocks of
// 16 columns: errors against 64 bits, relative to the result, 2.1e-7 -> 1.0e-7 at K 2,048 and 3.0e-7 -> 1.5e-7 at 8,192;
// of a 700-token prompt's logits at the Llama-3.2-1B shape 4.2e-7 -> 3.9e-7.)
#include "common.h"
#include "device.h"
#include "split_f32.h"
#include "tile_stream.h"

// columns of a span: 256, doubled until there are no more than 16; 128 of short sums, which have few spans to share
__host__ __device__ static inline int span_width(int K) {
  int w = K <= 1024 ? 128 : 256;
  while ((long)w * 16 < K) w <<= 1;
  return w;
}

// ===========================================================================
// Few rows of x (M <= 16, a decode step): bound by reading W once, and next to that by the instructions that split W and
// x, 52 and 44 for the 2 KB of W that a wave multiplies at a time. A workgroup owns ROWS rows of W; its waves take the spans, and the
// spans' sums meet in LDS.
//
// ROWS 16: A is 16 rows of W x a block of 32 columns, two load instructions that read 64 bytes of each row; B the same
// columns of 16 rows of x, from L2.
// ROWS 8: with at most 8 rows of x half of such a tile would be empty, so the tile holds two blocks of the same 8 rows
// (lanes ln < 8 the first, ln >= 8 the second), of W and of x alike. The products that matter are then D[n < 8][m < 8]
// and D[n >= 8][m >= 8], and every load instruction, of W and of x, still brings 1 KB that is used. It gives twice
// the workgroups. MT tiles of 8 rows of x share the loads of W.
//
// gemm_f32_few_kernel reads x again for every tile and takes the sums of any length;
// gemm_f32_held_kernel keeps x in registers and walks several tiles.
//
// Measured (one MI355X, cold weights, us at 4 and 16 rows; in brackets on the float32 matrix instructions): 16,384 x 2,048 26.3
// = 5.1 TB/s, 33.5 (25.8, 34.0), 2,048 x 8,192 18.5 = 3.6 TB/s, 27.7 (16.8, 29.9), 128,256 x 2,048 168 = 6.3 TB/s, 214
// (166, 228), 2,048 x 2,048 8.8, 10.0 (8.9, 10.2); the product of a decode step of 4 rows at the Llama-3.2-1B shape together 1 % more.
// ===========================================================================

// A tile's results from the spans' sums in LDS ([span][MT][64 lanes][4], lane and element as in D; of 8-row tiles
// the two halves).
template <int ROWS, int MT>
__device__ __forceinline__ void few_results(float* __restrict__ y, const float* __restrict__ x, const float* __restrict__ w,
                                            const float* sums, int spans, int M, int N, int K, int n0, long ldx, long ldy) {
  static_assert(ROWS * ROWS * MT % 64 == 0, "whole waves");
  for (int i = threadIdx.x; i < ROWS * ROWS * MT; i += blockDim.x) {
    const int n = i % ROWS, m = i / ROWS, t = m / ROWS, j = m % ROWS;
    const bool there = m < M && n0 + n < N;
    const float* p = sums + t * 256 + ((n >> 2) * 16 + j) * 4 + (n & 3);
    float s = 0.f;
    for (int sp = 0; sp < spans; ++sp, p += MT * 256) s += p[0];
    const bool odd = there && !is_finite(s);
    if (__builtin_expect(__any(odd), 0)) {
      bool nan_x = false;
      s = plain_dots<1>(s, odd, x + (size_t)m * ldx, w + (size_t)(n0 + n) * K, K, nan_x);
    }
    if (there) y[(size_t)m * ldy + n0 + n] = s;
  }
}

// What becomes of a tile's results. FORM_PLAIN: rows of y. The other two have 8-row tiles of four pairs of rows of W, the
// first of a pair in row n, the second in row n + 4, and finish the pair: FORM_GLU a gate and its up row, I apart,
// act(gate) * up; FORM_QKV rows j and j + D / 2 of a head of q | k | v, rotated (pairs, angles and cache pages as
// rope.hip has them). A decode step of 4 rows at the Llama-3.2-1B shape had a kernel of 4.7 us for either in every layer.
enum { FORM_PLAIN = 0, FORM_GLU = 1, FORM_QKV = 2 };

struct FewOut {
  int half;                        // FORM_GLU: I, FORM_QKV: D / 2
  int act;
  const int32_t *positions, *slots;          // of the rows of x; slots null: nothing goes into the cache
  const float* inv_freq;           // null: no rotation
  float *k_cache, *v_cache;
  int Hq, Hkv, page_size;
};

// row of W in place r (0 .. 7) of a tile
template <int FORM, int ROWS> __device__ __forceinline__ int few_row(const FewOut& o, int tile, int r, int N) {
  if (FORM == FORM_PLAIN) return min(ROWS * tile + r, N - 1);
  const int pair = 4 * tile + (r & 3);
  if (FORM == FORM_GLU) return pair + (r >= 4 ? o.half : 0);
  const int head = pair / o.half;
  return head * o.half + pair + (r >= 4 ? o.half : 0);
}

// The pairs of an 8-row tile from the spans' sums, added up as few_results does.
template <int FORM>
__device__ __forceinline__ void pair_results(float* __restrict__ y, const float* __restrict__ x, const float* __restrict__ w,
                                             const float* sums, int spans, int M, int N, int K, int tile, long ldx, long ldy,
                                             const FewOut& o) {
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));                  // (what follows of it is worked out here, for every tile: see plain_dots)
  if (tid < 64) {                                // (the first wave, half of it with a pair each)
    const int n = tid & 3, m = (tid >> 2) & 7;
    const bool there = tid < 32 && m < M;
    const float *p = sums + m * 4 + n, *p2 = p + 16 * 4;
    float a = 0.f, b = 0.f;
    for (int sp = 0; sp < spans; ++sp, p += 256, p2 += 256) {
      a += p[0];
      b += p2[0];
    }
    if (__builtin_expect(__any(there && !(is_finite(a) && is_finite(b))), 0)) {
      bool nan_x = false;
#pragma unroll 1
      for (int side = 0; side < 2; ++side) {
        const float v = side ? b : a;
        const float again = plain_dots<1>(v, there && !is_finite(v), x + (size_t)m * ldx,
                                       w + (size_t)few_row<FORM, 8>(o, tile, n + 4 * side, N) * K, K, nan_x);
        if (side) b = again; else a = again;
      }
    }
    if (!there) return;
    const int pair = 4 * tile + n;
    if (FORM == FORM_GLU) {
      y[(size_t)m * ldy + pair] = glu_act(o.act, a) * b;
    } else {
      const int head = pair / o.half, j = pair - head * o.half, D = 2 * o.half;
      if (o.inv_freq && head < o.Hq + o.Hkv) {
        float s, c;
        sincosf((float)o.positions[m] * o.inv_freq[j], &s, &c);
        const float x1 = a, x2 = b;
        a = x1 * c - x2 * s;
        b = x2 * c + x1 * s;
      }
      float* at = nullptr;
      if (head < o.Hq) {
        at = y + (size_t)m * ldy + (size_t)head * D;
      } else {
        const int slot = o.slots ? o.slots[m] : -1;
        const bool k = head < o.Hq + o.Hkv;
        if (slot >= 0) {
          const int page = slot / o.page_size, off = slot - page * o.page_size, h = head - o.Hq - (k ? 0 : o.Hkv);
          at = (k ? o.k_cache : o.v_cache) + (((size_t)page * o.Hkv + h) * o.page_size + off) * D;
        }
      }
      if (at) {
        at[j] = a;
        at[j + o.half] = b;
      }
    }
  }
}

// Where a lane's columns of x begin, and the column from there of load u: two loads make the eight columns a lane has of
// a fragment, of 16-row tiles one block, of 8-row tiles two, the first in the lanes ln < 8.
template <int ROWS> __device__ __forceinline__ int few_first(int ln, int lg) { return 4 * lg + (ROWS == 8 ? 32 * (ln >> 3) : 0); }
template <int ROWS> __host__ __device__ constexpr int few_column(int u) { return (ROWS == 8 ? 64 : 32) * (u / 2) + 16 * (u % 2); }

// The same of W. In 8-row tiles a load takes whole 128-byte lines, a block of all 8 rows (with the columns of x, half of
// two blocks, it is 15 % slower: 128,256 x 2,048 164 -> 195 us): its second half comes to the lanes ln >= 8,
// and few_pair hands the halves over.
template <int ROWS> __device__ __forceinline__ int few_first_w(int ln, int lg) { return 4 * lg + (ROWS == 8 ? 16 * (ln >> 3) : 0); }
template <int ROWS> __host__ __device__ constexpr int few_column_w(int u) { return (ROWS == 8 ? 32 : 16) * u; }

// the lower (upper) half of every 16 lanes from ``here``, the other from the lanes 8 away of ``there``
template <bool LOWER> __device__ __forceinline__ uint32_t half_of(uint32_t here, uint32_t there) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)here, (int)there, 0x128, 0xf, LOWER ? 0xc : 0x3, false);
}
template <int ROWS> __device__ __forceinline__ Split few_pair(const F4& a, const F4& b) {
  if (ROWS == 16) return split8(a, b);
  F4 first, second;
  first.u = make_uint4(half_of<true>(a.u.x, b.u.x), half_of<true>(a.u.y, b.u.y), half_of<true>(a.u.z, b.u.z),
                       half_of<true>(a.u.w, b.u.w));
  second.u = make_uint4(half_of<false>(b.u.x, a.u.x), half_of<false>(b.u.y, a.u.y), half_of<false>(b.u.z, a.u.z),
                        half_of<false>(b.u.w, a.u.w));
  return split8(first, second);
}

// acc += a fragment's products. Of 8-row tiles D[n < 8][m < 8] is the sum of the fragment's first block and
// D[n >= 8][m >= 8], 40 lanes on, that of the second: added one after the other, in the lanes of the first.
template <int ROWS> __device__ __forceinline__ void few_add(f32x4_t& acc, const Split& w, const Split& x) {
  const f32x4_t t = split_dot(w, x);
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] += t[i];
  if (ROWS == 8) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const auto other = __builtin_amdgcn_permlane32_swap(__float_as_uint(t[i]), __float_as_uint(t[i]), false, false);
      acc[i] += __uint_as_float(__builtin_amdgcn_update_dpp(0, other[1], 0x128, 0xf, 0xf, true));   // (rotate by 8 of 16)
    }
  }
}

// R fragments of W and of x are under way, and come in the order in which they are used. (x asked for first and split while
// W is on its way: 2,048 x 8,192 18.4 -> 20.7.)
template <int ROWS, int MT, int R, int FORM>
__global__ void __launch_bounds__(1024)
gemm_f32_few_kernel(float* __restrict__ y, const float* __restrict__ x, const float* __restrict__ w,
                    int M, int N, int K, long ldx, long ldy, int width, FewOut out) {
  extern __shared__ float red[];                 // [waves][MT][64][4]: a wave a span
  static_assert((ROWS == 16 && MT == 1) || ROWS == 8, "rows of W a tile");
  static_assert(FORM == FORM_PLAIN || (ROWS == 8 && MT == 1), "pairs lie in 8-row tiles, of up to 8 rows of x");
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, ln = lane & 15, lg = lane >> 4;
  const int kb = wave * width, ke = min(K, kb + width);
  const int kx = kb + few_first<ROWS>(ln, lg), kw = kb + few_first_w<ROWS>(ln, lg);
  const float* wp = w + (size_t)few_row<FORM, ROWS>(out, blockIdx.x, ln % ROWS, N) * K + kw;
  const float* xp[MT];
  int x_end[MT];                                 // (0: no row of x)
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = ROWS * t + ln % ROWS;
    x_end[t] = m < M ? ke : 0;
    xp[t] = x + (size_t)min(m, M - 1) * ldx + kx;
  }
  f32x4_t acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  constexpr int FB = few_column<ROWS>(2);        // columns of a fragment
  F4 wr[R][2], xr[R][MT][2];
  auto load_w = [&](int r, int k) __attribute__((always_inline)) {     // k: from kb on
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int at = k + few_column_w<ROWS>(u);
      wr[r][u].u = kw + at < ke ? load_once(wp + at) : zero16();
    }
  };
  auto load_x = [&](int r, int k) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int at = k + few_column<ROWS>(u);
        xr[r][t][u].u = kx + at < x_end[t] ? load16(xp[t] + at) : zero16();
      }
  };
  const int fragments = max(0, (ke - kb + FB - 1) / FB);
  auto load = [&](int r, int f) __attribute__((always_inline)) {
    load_w(r, FB * f);
    load_x(r, FB * f);
  };
#pragma unroll
  for (int r = 0; r < R; ++r) load(r, r);
  for (int f = 0; f < fragments; f += R) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (f + r >= fragments) break;
      const Split s = few_pair<ROWS>(wr[r][0], wr[r][1]);
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        few_add<ROWS>(acc[t], s, split8(xr[r][t][0], xr[r][t][1]));
        // (one fragment's parts at a time: there are no registers for more)
        asm volatile("" : "+v"(acc[t]));
      }
      if (f + r + R < fragments) load(r, f + r + R);
    }
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) *reinterpret_cast<f32x4_t*>(red + (((size_t)wave * MT + t) * 64 + lane) * 4) = acc[t];
  __syncthreads();
  if (FORM == FORM_PLAIN) few_results<ROWS, MT>(y, x, w, red, blockDim.x >> 6, M, N, K, blockIdx.x * ROWS, ldx, ldy);
  else pair_results<FORM>(y, x, w, red, blockDim.x >> 6, M, N, K, blockIdx.x, ldx, ldy, out);
}

// Up to 8 rows (16 of 16-row tiles) with a wave's share of the columns in registers: x [ROWS, KB NB] of every wave
// is read once, and the workgroup then walks ROWS-row tiles of W (blockIdx.x, + gridDim.x, ...), so that W is all that
// is read in the loop: read again for every tile, x comes through the same path from L2 as W does and is as many
// bytes (128,256 x 2,048, us at 1, 4 and 8 rows: 185, 214, 254; held 161, 171, 177). The next tile's first columns are on their way while a tile's
// sums are added up, in two buffers, one barrier a tile. SB: load blocks of a span.
#define RING 2
template <int ROWS, int NB, int SB, int FORM>
__global__ void __launch_bounds__(1024)
gemm_f32_held_kernel(float* __restrict__ y, const float* __restrict__ x, const float* __restrict__ w,
                     int M, int N, int K, long ldx, long ldy, int tiles, FewOut out) {
  static_assert(ROWS == 8 || FORM == FORM_PLAIN, "pairs lie in 8-row tiles");
  constexpr int KB = ROWS == 8 ? 32 : 16;        // columns of a load, of all lanes
  constexpr int F = NB / 2, R = NB > 8 ? RING : 4;   // fragments (two loads) a tile, and under way
  constexpr int EACH = NB / SB;                  // spans of a wave
  static_assert(F % R == 0, "a tile's fragments come into the same registers as the last tile's");
  static_assert(NB % SB == 0 && SB % 2 == 0, "a wave's share ends with a span, a span with a fragment");
  extern __shared__ float red[];                 // [2][waves][EACH][64][4]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, ln = lane & 15, lg = lane >> 4;
  const int nwaves = blockDim.x >> 6;
  const int kb = KB * NB * wave + few_first<ROWS>(ln, lg), kw = KB * NB * wave + few_first_w<ROWS>(ln, lg);
  const int left = K - kb, left_w = K - kw;      // this lane's columns of load b are there if few_column(b) < left
  F4 xf[NB];
  {
    const float* xp = x + (size_t)min(ln % ROWS, M - 1) * ldx + kb;
    const bool row = ln % ROWS < M;
#pragma unroll
    for (int b = 0; b < NB; ++b) xf[b].u = row && few_column<ROWS>(b) < left ? load16(xp + few_column<ROWS>(b)) : zero16();
  }
  F4 ring[R][2];
  const float* wp = w + (size_t)few_row<FORM, ROWS>(out, blockIdx.x, ln % ROWS, N) * K + kw;
  auto load_w = [&](F4 (&to)[2], int f) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int at = few_column_w<ROWS>(2 * f + u);
      to[u].u = at < left_w ? load_once(wp + at) : zero16();
    }
  };
#pragma unroll
  for (int f = 0; f < R; ++f) load_w(ring[f], f);
  int at = 0;
  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x, at ^= 1) {
    float* const sums = red + at * nwaves * EACH * 256;
    const bool more = tile + (int)gridDim.x < tiles;
    f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int f = 0; f < F; ++f) {
      Split s = few_pair<ROWS>(ring[f % R][0], ring[f % R][1]);
      // (the parts take other registers: the next loads go to those that have become free)
      asm volatile("" : "+v"(s.h.u.x), "+v"(s.h.u.y), "+v"(s.h.u.z), "+v"(s.h.u.w), "+v"(s.m.u.x), "+v"(s.m.u.y),
                   "+v"(s.m.u.z), "+v"(s.m.u.w), "+v"(s.l.u.x), "+v"(s.l.u.y), "+v"(s.l.u.z), "+v"(s.l.u.w));
      if (f + R < F) {
        load_w(ring[f % R], f + R);
      } else {
        if (f + R == F) wp = w + (size_t)few_row<FORM, ROWS>(out, min(tile + (int)gridDim.x, tiles - 1), ln % ROWS, N) * K + kw;
        if (more) load_w(ring[f % R], f + R - F);
      }
      // (x is split anew for every tile, and here: kept, or done at once, the parts of NB > 8 loads would not fit into the
      // registers)
      if (NB > 8)
#pragma unroll
        for (int u = 2 * f; u < 2 * f + 2; ++u)
          asm volatile("" : "+v"(xf[u].u.x), "+v"(xf[u].u.y), "+v"(xf[u].u.z), "+v"(xf[u].u.w));
      few_add<ROWS>(acc, s, split8(xf[2 * f], xf[2 * f + 1]));
      if (NB > 8) asm volatile("" : "+v"(acc));
      if ((2 * f + 2) % SB == 0) {               // the end of a span
        *reinterpret_cast<f32x4_t*>(sums + ((wave * EACH + 2 * f / SB) * 64 + lane) * 4) = acc;
        acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    }
    tile_wait_lds();
    tile_meet();                                 // (the loads of the next tile stay under way)
    if (FORM == FORM_PLAIN) few_results<ROWS, 1>(y, x, w, sums, nwaves * EACH, M, N, K, ROWS * tile, ldx, ldy);
    else pair_results<FORM>(y, x, w, sums, nwaves * EACH, M, N, K, tile, ldx, ldy, out);
  }
}

// Tiles of ``rows`` rows of W, x held in registers (up to 8 rows and 8,192 columns, or 16 and 4,096) where a workgroup
// walks several of them; where every workgroup has one, x is read no more often by the other kernel, which has twice as many
// loads of W under way (2,048 x 8,192, 4 rows, 19.1 us held, 18.4 so).
template <int FORM>
static int launch_few(float* y, const float* x, const float* w, int M, int N, int K, long ldx, long ldy, int rows,
                      const FewOut& out, hipStream_t st) {
  const int cus = compute_units();
  const long blocks = (N + rows - 1) / rows;
  const int width = span_width(K), spans = (K + width - 1) / width;
  const bool half = rows == 8 && K <= 4096;      // (256 columns a wave)
  const int share = rows == 8 && !half ? 512 : 256;
  const int waves = (K + share - 1) / share;
  const bool holds = rows == 8 ? M <= 8 && K <= 8192 : K <= 4096;
  const long resident = holds ? (long)cus * (16 / waves) : 0;
  const long walk = holds ? (blocks + resident - 1) / resident : 1;
#define GO(ROWS, MT, FORM)                                                                                            \
  gemm_f32_few_kernel<ROWS, MT, 4 / MT, FORM><<<(unsigned)blocks, spans * 64, (size_t)spans * MT * 1024, st>>>(       \
      y, x, w, M, N, K, ldx, ldy, width, out)
  if (!holds || (rows == 8 && walk == 1)) {
    if (rows == 16) GO(16, 1, FORM_PLAIN);
    else if (M <= 8) GO(8, 1, FORM);
    else GO(8, 2, FORM_PLAIN);
    return ptl_launch_status();
  }
#undef GO
  const unsigned grid = (unsigned)((blocks + walk - 1) / walk);
#define HELD(ROWS, NB, SB)                                                                                      \
  gemm_f32_held_kernel<ROWS, NB, SB, ROWS == 8 ? FORM : FORM_PLAIN>                                             \
      <<<grid, waves * 64, (size_t)waves * (NB / SB) * 2048, st>>>(y, x, w, M, N, K, ldx, ldy, (int)blocks, out)
  if (rows == 16 && width == 128) HELD(16, 16, 8);
  else if (rows == 16) HELD(16, 16, 16);
  else if (half && width == 128) HELD(8, 8, 4);
  else if (half) HELD(8, 8, 8);
  else HELD(8, 16, 16);
#undef HELD
  return ptl_launch_status();
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// M <= 16, K % 4 == 0, ldx % 4 == 0, x and w 16-byte aligned.
extern "C" int ptl_gemm_f32_few(float* y, const float* x, const float* w, int M, int N, int K, long ldx, long ldy,
                                hipStream_t st) {
  if (M <= 0 || N <= 0) return PTL_OK;
  if (M > 16 || K <= 0 || K % 4 || (M > 1 && ldx % 4) || ldx < K || ldy < N || !aligned16(x) || !aligned16(w))
    return PTL_ERR_ARG;
  // up to 8 rows 8-row tiles; beyond, where they cost a second load of x, only while 16-row tiles leave a third of
  // the compute units empty (us at 16 rows, 8- against 16-row tiles: 2,048 x 8,192 29 / 37, 3,072 x 2,048 16.2 /
  // 11.9, 16,384 x 2,048 54.6 / 39.9). At 32 rows gemm_f32_few_kernel is slower than the tiles below at every size.
  const int cus = compute_units();
  const int rows = M <= 8 || (N + 15) / 16 * 3 < 2L * cus ? 8 : 16;
  // (16 rows, read again against held: 16,384 x 2,048 43 / 36, 128,256 x 2,048 317 / 230)
  return launch_few<FORM_PLAIN>(y, x, w, M, N, K, ldx, ldy, rows, FewOut{}, st);
}

static bool pairs_ok(int M, int K, long ldx, const float* x, const float* w) {
  return M > 0 && M <= 8 && K > 0 && K <= 8192 && K % 4 == 0 && (M == 1 || ldx % 4 == 0) && ldx >= K && aligned16(x) && aligned16(w);
}

// out [M, I] = act(x Wg^T) * (x Wu^T) for W = [Wg; Wu] [2 I, K]: up to 8 rows, K up to 8,192 in steps of 4, I in steps of 4.
extern "C" int ptl_gate_up_f32(float* out, const float* x, const float* w, int M, int I, int K, long ldx, int act,
                               hipStream_t st) {
  if (!pairs_ok(M, K, ldx, x, w) || I <= 0 || I % 4 || (act != GLU_SILU && act != GLU_GELU_TANH)) return PTL_ERR_ARG;
  FewOut o{};
  o.half = I;
  o.act = act;
  return launch_few<FORM_GLU>(out, x, w, M, 2 * I, K, ldx, I, 8, o, st);
}

// q | k | v = x W^T, q and k rotated; q to q_out [M, Hq D], k and v into the cache pages at ``slots`` (null: nowhere).
// Up to 8 rows, K up to 8,192 in steps of 4, D in steps of 8.
extern "C" int ptl_qkv_rope_store_f32(float* q_out, const float* x, const float* w, int M, int K, long ldx,
                                      const int32_t* positions, const float* inv_freq, const int32_t* slots,
                                      float* k_cache, float* v_cache, int Hq, int Hkv, int D, int page_size,
                                      hipStream_t st) {
  if (!pairs_ok(M, K, ldx, x, w) || Hq <= 0 || Hkv <= 0 || D <= 0 || D % 8 || page_size <= 0 || !positions ||
      (slots && (!k_cache || !v_cache)))
    return PTL_ERR_ARG;
  return launch_few<FORM_QKV>(q_out, x, w, M, (Hq + 2 * Hkv) * D, K, ldx, (long)Hq * D, 8,
                               FewOut{D / 2, 0, positions, slots, inv_freq, k_cache, v_cache, Hq, Hkv, page_size}, st);
}

// ===========================================================================
// Many rows of x (a prompt portion), both forms with the order of sums of the kernels above. Where K is a multiple of
// 32, gemm_f32_stream_kernel: a first kernel splits x into its parts, and waves that do nothing else bring them and W through
// LDS (tile_stream.h); else, and for small products, gemm_f32_tile_kernel (split_f32.h), which splits x itself.
//
// A grid of few tiles is cut along K as well (a number of spans a workgroup): the spans' sums go to a workspace
// [spans, M, N] and another kernel adds them in order.
//
// Measured (one MI355X, cold weights, us, with the kernel that splits x; in brackets tiles of 64 x 64 on the float32 matrix
// instructions, which ran before): 700 x 16,384 x 2,048 240 = 196 TFLOP/s (472), 700 x 2,048 x 8,192 146 (237), 700 x 3,072 x
// 2,048 77 (110), 483 x 4,096 x 2,048 57 (94), 64 x 2,048 x 8,192 27 (30), 17 x 2,048 x 2,048 13.5 (13.1).
// ===========================================================================

// The results of a wave's tile that are not finite, made again: it has stored TM groups of 16 rows of x, from m0 on, and TN4
// results a lane and group, of rows n0 + 16 (e / 4) + 4 lg + e % 4 of W; bit i of odd: one of this lane's results in group i.
template <int TN4, int TM>
__device__ __forceinline__ void tile_again(float* __restrict__ y, long ldy, unsigned odd, int m0, int n0, int M, int N,
                                           const float* __restrict__ x, long ldx, const float* __restrict__ w, int K) {
  const int lane = threadIdx.x & 63, ln = lane & 15, lg = lane >> 4;
  if (__builtin_expect(!__any(odd), 1)) return;
#pragma unroll 1
  for (int i = 0; i < TM; ++i) {
    if (!__any(odd >> i & 1)) continue;
    const int m = m0 + 16 * i + ln;
    const float* xr = x + (size_t)min(m, M - 1) * ldx;
    bool nan_x = false;
#pragma unroll 1
    for (int e = 0; e < TN4; ++e) {
      const int n = n0 + 16 * (e >> 2) + 4 * lg + (e & 3);
      const bool there = m < M && n < N && (odd >> i & 1);
      float* at = y + (size_t)m * ldy + n;
      const float v = there ? *at : 0.f;         // (as this lane has stored it)
      const bool again = there && !is_finite(v);
      if (!__any(again)) continue;
      const float s = plain_dots(v, again, xr, w + (size_t)min(n, N - 1) * K, K, nan_x);
      if (again) *at = s;
    }
  }
}

// K not a multiple of 32, or small products: tile_plan (700 x 16,384 x 2,048 320 us in this form).
template <int TA, int TC, bool PARTS>
__global__ void __launch_bounds__(256, 2)
gemm_f32_tile_kernel(float* __restrict__ y, const float* __restrict__ x, const float* __restrict__ w,
                     int M, int N, int K, long ldx, long ldy, int tiles_m, int tiles, int width, int k_per_split,
                     float* __restrict__ parts) {
  constexpr int TN = 64 * TA, TM = 16 * TC, EACH = SplitX<TC>::EACH;
  __shared__ uint4 lds[SplitX<TC>::LDS];
  // Workgroups go to the eight XCDs in turn: each gets a run of tiles, neighbours in the run share
  // rows of W, so that W comes into one L2 once.
  const int per_xcd = (tiles + 7) / 8;
  const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (tile >= tiles || (int)(blockIdx.x >> 3) >= per_xcd) return;
  const int n0 = tile / tiles_m * TN, m0 = tile % tiles_m * TM;
  const int kb = blockIdx.y * k_per_split, ke = min(K, kb + k_per_split);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, ln = lane & 15, lg = lane >> 4;
  const int wn = n0 + 16 * TA * wave;
  const float* wp[TA];
  const float* xp[EACH];
#pragma unroll
  for (int a = 0; a < TA; ++a) wp[a] = w + (size_t)min(wn + 16 * a + ln, N - 1) * K;
#pragma unroll
  for (int i = 0; i < EACH; ++i) xp[i] = x + (size_t)min(m0 + (int)(threadIdx.x >> 2) + 64 * i, M - 1) * ldx;
  // results [M, N] of row stride ld, from D[n = 4 lg + i][m = ln] of every 16 x 16 tile
  auto store = [&](float* to, long ld, const f32x4_t (&v)[TA][TC]) __attribute__((always_inline)) {
    const bool four = (N & 3) == 0 && (ld & 3) == 0 && (reinterpret_cast<uintptr_t>(to) & 15) == 0;
    unsigned odd = 0;                            // groups of 16 rows of x with a result that is not finite
#pragma unroll
    for (int c = 0; c < TC; ++c) {
      const int m = m0 + 16 * c + ln;
      if (m >= M) continue;
#pragma unroll
      for (int a = 0; a < TA; ++a) {
        const int n = wn + 16 * a + 4 * lg;
        float* at = to + (size_t)m * ld + n;
        if (four) {
          if (n < N) *reinterpret_cast<f32x4_t*>(at) = v[a][c];
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (n + i < N) at[i] = v[a][c][i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) odd |= is_finite(v[a][c][i]) ? 0u : 1u << c;
      }
    }
    return odd;
  };
  f32x4_t acc[TA][TC], sum[TA][TC];              // of the span, of the spans so far
#pragma unroll
  for (int a = 0; a < TA; ++a)
#pragma unroll
    for (int c = 0; c < TC; ++c) acc[a][c] = sum[a][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  split_tile<TA, TC>(lds, wp, xp, kb, ke, width, acc, [&](int k) __attribute__((always_inline)) {
    if (PARTS) {
      store(parts + (size_t)(k / width) * M * N, N, acc);
    } else {
#pragma unroll
      for (int a = 0; a < TA; ++a)
#pragma unroll
        for (int c = 0; c < TC; ++c)
#pragma unroll
          for (int i = 0; i < 4; ++i) sum[a][c][i] += acc[a][c][i];
    }
#pragma unroll
    for (int a = 0; a < TA; ++a)
#pragma unroll
      for (int c = 0; c < TC; ++c) acc[a][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  });
  if (!PARTS) tile_again<4 * TA, TC>(y, ldy, store(y, ldy, sum), m0, wn, M, N, x, ldx, w, K);
}

__global__ void __launch_bounds__(256)
gemm_f32_sum_kernel(float* __restrict__ y, const float* __restrict__ parts, int spans, const float* __restrict__ x,
                    const float* __restrict__ w, int M, int N, int K, long ldx, long ldy) {
  const long total = (long)M * N;
  const bool four = (N & 3) == 0 && (ldy & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
  const long first = four ? ((long)blockIdx.x * 256 + threadIdx.x) * 4 : (long)blockIdx.x * 1024 + threadIdx.x;
  const int step = four ? 1 : 256;               // a thread has four results, ``step`` apart
  f32x4_t s = {0.f, 0.f, 0.f, 0.f};
  if (four) {
    if (first < total)
#pragma unroll 4
      for (int p = 0; p < spans; ++p) s += *reinterpret_cast<const f32x4_t*>(parts + (size_t)p * total + first);
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (first + j * step < total)
        for (int p = 0; p < spans; ++p) s[j] += parts[(size_t)p * total + first + j * step];
  }
  if (__builtin_expect(__any(!(is_finite(s[0]) && is_finite(s[1]) && is_finite(s[2]) && is_finite(s[3]))), 0)) {
    bool nan_x = false;
    long last = -1;
#pragma unroll 1
    for (int j = 0; j < 4; ++j) {
      const long i = first + j * step;
      const float v = j == 0 ? s[0] : j == 1 ? s[1] : j == 2 ? s[2] : s[3];
      const bool odd = i < total && !is_finite(v);
      const long m = odd ? i / N : 0, n = odd ? i % N : 0;
      if (m != last) nan_x = false;
      last = m;
      const float again = plain_dots(v, odd, x + m * ldx, w + n * K, K, nan_x);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = e == j ? again : s[e];
    }
  }
  if (four) {
    if (first < total) *reinterpret_cast<f32x4_t*>(y + first / N * ldy + first % N) = s;
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const long i = first + j * step;
      if (i < total) y[i / N * ldy + i % N] = s[j];
    }
  }
}

// The parts of x for gemm_f32_stream_kernel: [blocks of 32 columns][rows: h | m, 128 bytes][pairs of rows: l | l, 128 bytes],
// rows of 128 bytes as tile_stream.h has them. One thread eight columns.
__host__ __device__ static inline size_t split_rows_bytes(int Mp) { return (size_t)Mp * 192; }

__global__ void __launch_bounds__(256)
split_rows_kernel(unsigned char* __restrict__ out, const float* __restrict__ x, int M, int K, long ldx, int Mp) {
  const int lg = threadIdx.x & 3, row = blockIdx.x * 64 + (threadIdx.x >> 2), b = blockIdx.y;
  if (row >= M) return;
  const float* p = x + (size_t)row * ldx + 32 * b + 4 * lg;
  F4 u, v;
  u.u = load16(p);
  v.u = load16(p + 16);
  const Split s = split8(u, v);
  unsigned char* at = out + split_rows_bytes(Mp) * b;
  *reinterpret_cast<uint4*>(at + (size_t)row * 128 + 16 * lg) = s.h.u;
  *reinterpret_cast<uint4*>(at + (size_t)row * 128 + 64 + 16 * lg) = s.m.u;
  *reinterpret_cast<uint4*>(at + (size_t)Mp * 128 + (size_t)row * 64 + 16 * lg) = s.l.u;
}

struct StreamArgs {
  float *y, *parts;               // parts: of the spans, where K is cut
  const float *x, *w;
  const unsigned char* xs;
  int M, N, K, Mp;
  long ldx, ldy;
  int tiles_m, tiles_n, splits, per, width;
  int act;
};

// What becomes of a tile's sums: y; parts, the sums of every span by itself; or, for W = [Wg; Wu] with N rows each, act(gate) * up,
// the rows of a wave being 16 of Wg and the same 16 of Wu: the two are finished where they are, where the product of 700 rows and
// 2 x 8,192 of 2,048 columns wrote 46 MB for a kernel of 16 us that read them again (with it 9.33, so 9.11 ms for such a prompt
// through 16 layers).
enum { STREAM_Y = 0, STREAM_PARTS = 1, STREAM_GLU = 2 };

// Tiles of BM rows of x and BN of W; four waves multiply, each all rows of x and a quarter of W's, PW bring the operands, a block
// of 32 columns at a time into one of NB buffers. W lies in LDS as it is in memory and is split by the wave that
// wants it, a block ahead, between the products of the block before: 11 instructions for a pair of
// numbers, where every matrix instruction leaves room for about one. The sums of a 16 x 16 tile are added
// while the next tile's are on their way. What bounds it: a block of 128 x 128 takes 0.98 us a workgroup where 96 matrix instructions
// of 18 clocks take 0.72, and 1.23 with all compute units at work, 40 KB from L2 each. (Without the
// order by hand the compiler moves the splitting and the sums behind all products of the block: 1.11 us; with two
// loading waves 700 x 16,384 x 2,048 takes 284 us, with four 240; x split by every workgroup 308 at best.)
template <int BM, int BN, int NB, int PW, int MODE>
__global__ void __launch_bounds__(64 * (4 + PW))
gemm_f32_stream_kernel(const StreamArgs a) {
  constexpr bool PARTS = MODE == STREAM_PARTS, GLU = MODE == STREAM_GLU;
  constexpr int COLS = GLU ? BN / 2 : BN;        // columns of y a tile gives
  static_assert(!GLU || BN == 128, "a wave has 16 rows of either");
  constexpr int TM = BM / 16, TN = BN / 64;
  constexpr int ROWS = BN + BM + BM / 2, CHUNK = ROWS * TILE_ROW;
  extern __shared__ __align__(16) unsigned char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int M = a.M, N = a.N, K = a.K;
  const int total = a.tiles_m * a.tiles_n * a.splits, G = gridDim.x;
  const int run = G >> 3, rest = G & 7, xcd = blockIdx.x & 7;
  const int first_tile = xcd * run + min(xcd, rest) + (blockIdx.x >> 3);
  const int my_tiles = (total - first_tile + G - 1) / G;
  auto place = [&](int t, int& m0, int& n0, int& kb, int& chunks) __attribute__((always_inline)) {
    const int each = a.tiles_m * a.tiles_n, split = t / each, u = t - split * each;
    const int tn = u / a.tiles_m;
    n0 = tn * COLS;
    m0 = (u - tn * a.tiles_m) * BM;
    kb = split * a.per;
    chunks = (min(K, kb + a.per) - kb) / SPLIT_BK;
  };

  if (wave >= 4) {
    constexpr int LI = ROWS / 8 / PW;
    static_assert(ROWS % (8 * PW) == 0 && (NB - 2) * LI < 64, "loads are counted in six bits");
    const int lrow = lane >> 3, lpiece = (lane & 7) ^ lrow, first = (wave - 4) * LI;
    const char* src[LI];
    const long xstep = (long)split_rows_bytes(a.Mp);
    int all = 0, m0, n0, kb, chunks;
    for (int n = 0; n < my_tiles; ++n) { place(first_tile + n * G, m0, n0, kb, chunks); all += chunks; }
    int next = 0, next_tile = 0, left = 0, slot = 0;
    auto fetch = [&]() __attribute__((always_inline)) {
      if (left == 0) {
        place(first_tile + next_tile * G, m0, n0, kb, left);
        ++next_tile;
        const unsigned char* xb = a.xs + (size_t)(kb / SPLIT_BK) * xstep;
#pragma unroll
        for (int i = 0; i < LI; ++i) {
          const int r = 8 * (first + i) + lrow;
          const char* p;
          if (8 * (first + i) < BN) {
            const int row = GLU ? min(n0 + 16 * (r >> 5) + (r & 15), N - 1) + (r & 16 ? N : 0) : min(n0 + r, N - 1);
            p = reinterpret_cast<const char*>(a.w + (size_t)row * K + kb);
          }
          else if (8 * (first + i) < BN + BM) p = reinterpret_cast<const char*>(xb + (size_t)(m0 + r - BN) * 128);
          else p = reinterpret_cast<const char*>(xb + (size_t)a.Mp * 128 + (size_t)(m0 / 2 + r - BN - BM) * 128);
          src[i] = p + 16 * lpiece;
        }
      }
      unsigned char* dst = lds + (size_t)slot * CHUNK + 1024 * first;
#pragma unroll
      for (int i = 0; i < LI; ++i) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src[i],
                                         (__attribute__((address_space(3))) void*)(dst + 1024 * i), 16, 0, 0);
        src[i] += 8 * (first + i) < BN ? (long)TILE_ROW : xstep;
      }
      ++next;
      --left;
      slot = slot + 1 == NB ? 0 : slot + 1;
    };
    for (int c = 0; c < NB - 1; ++c)
      if (next < all) fetch();
    for (int c = 0; c < all; ++c) {
      // chunks c and c + 1 have landed when at most the chunks after them are still under way
      switch (max(0, min(NB - 3, all - 2 - c))) {
        case 0: tile_wait_loads_but<0>(); break;
        case 1: tile_wait_loads_but<LI>(); break;
        default: tile_wait_loads_but<(NB > 4 ? 2 * LI : 0)>(); break;
      }
      tile_meet();                               // chunk c - 1 has been read
      if (next < all) fetch();
    }
    return;
  }

  const int ln = lane & 15, lg = lane >> 4;
  const int p0 = 16 * (lg ^ (ln & 7)), p1 = 16 * ((4 + lg) ^ (ln & 7));
  const int w_at = (wave * 16 * TN + ln) * TILE_ROW, x_at = (BN + ln) * TILE_ROW;
  const int l_at = (BN + BM + (ln >> 1)) * TILE_ROW + 16 * ((4 * (ln & 1) + lg) ^ ((ln >> 1) & 7));
  f32x4_t acc[TN][TM], sum[TN][TM];
  Split wa[TN], wb[TN];
  F4 wr[TN][2];
  Split x[2];
  auto read_x = [&](Split& to, const unsigned char* at, int i) __attribute__((always_inline)) {
    to.h.u = load16(at + x_at + i * 16 * TILE_ROW + p0);
    to.m.u = load16(at + x_at + i * 16 * TILE_ROW + p1);
    to.l.u = load16(at + l_at + i * 8 * TILE_ROW);
  };
  auto read_w = [&](const unsigned char* at) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      wr[j][0].u = load16(at + w_at + j * 16 * TILE_ROW + p0);
      wr[j][1].u = load16(at + w_at + j * 16 * TILE_ROW + p1);
    }
  };
  auto split_pair = [&](Split (&wn)[TN], int q) __attribute__((always_inline)) {        // q: 0 .. 4 TN - 1
    const int j = q >> 2, e = q & 3;
    const F4& f = wr[j][e >> 1];
    uint32_t h, m, l;
    split2(f.f[2 * (e & 1)], f.f[2 * (e & 1) + 1], h, m, l);
    (&wn[j].h.u.x)[e] = h;
    (&wn[j].m.u.x)[e] = m;
    (&wn[j].l.u.x)[e] = l;
  };
  int slot = 0;
  bool first = true;
  for (int n = 0; n < my_tiles; ++n) {
    int m0, n0, kb, chunks;
    place(first_tile + n * G, m0, n0, kb, chunks);
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[j][i] = sum[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto store = [&](float* to, long ld, const f32x4_t (&v)[TN][TM]) __attribute__((always_inline)) {
      const bool four = (N & 3) == 0 && (ld & 3) == 0 && (reinterpret_cast<uintptr_t>(to) & 15) == 0;
      unsigned odd = 0;                          // groups of 16 rows of x with a result that is not finite
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int m = m0 + 16 * i + ln;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int c = n0 + 16 * TN * wave + 16 * j + 4 * lg;
          float* at = to + (size_t)m * ld + c;
          if (four) {
            if (c < N) *reinterpret_cast<f32x4_t*>(at) = v[j][i];
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (c + e < N) at[e] = v[j][i][e];
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) odd |= is_finite(v[j][i][e]) ? 0u : 1u << i;
        }
      }
      return odd;
    };
    // one chunk; its weights' parts are in ws, those of the next go to wn
    auto chunk = [&](int c, Split (&ws)[TN], Split (&wn)[TN]) __attribute__((always_inline)) {
      tile_meet();
      const unsigned char* at = lds + (size_t)slot * CHUNK;
      slot = slot + 1 == NB ? 0 : slot + 1;
      const unsigned char* after = lds + (size_t)slot * CHUNK;
      if (first) {
        read_w(at);
#pragma unroll
        for (int q = 0; q < 4 * TN; ++q) split_pair(ws, q);
        first = false;
      }
      read_x(x[0], at, 0);
      read_w(after);                             // (behind the last chunk: what is there is not used)
      f32x4_t t[2][TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        __builtin_amdgcn_sched_barrier(0);
        if (i + 1 < TM) read_x(x[(i + 1) & 1], at, i + 1);
#pragma unroll
        for (int j = 0; j < TN; ++j) t[i & 1][j] = split_dot(ws[j], x[i & 1]);
        if (i > 0)
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[j][i - 1][e] += t[(i - 1) & 1][j][e];
#pragma unroll
        for (int q = 4 * TN * i / TM; q < 4 * TN * (i + 1) / TM; ++q) split_pair(wn, q);
        // (sums and parts are wanted here, between the products: the compiler would put them all behind the loop)
        if (i > 0)
#pragma unroll
          for (int j = 0; j < TN; ++j) asm volatile("" : "+v"(acc[j][i - 1]));
#pragma unroll
        for (int q = 4 * TN * i / TM; q < 4 * TN * (i + 1) / TM; ++q)
          asm volatile("" : "+v"((&wn[q >> 2].h.u.x)[q & 3]), "+v"((&wn[q >> 2].m.u.x)[q & 3]), "+v"((&wn[q >> 2].l.u.x)[q & 3]));
#pragma unroll
        for (int g = 0; g < 6 * TN; ++g) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (g < 3) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[j][TM - 1][e] += t[(TM - 1) & 1][j][e];
      if (c + 1 == chunks || (kb + (c + 1) * SPLIT_BK) % a.width == 0) {
        if (PARTS) store(a.parts + (size_t)((kb + c * SPLIT_BK) / a.width) * M * N, N, acc);
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int i = 0; i < TM; ++i) {
            if (!PARTS)
#pragma unroll
              for (int e = 0; e < 4; ++e) sum[j][i][e] += acc[j][i][e];
            acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
          }
      }
      tile_wait_lds();
    };
    for (int c = 0; c < chunks; c += 2) {
      chunk(c, wa, wb);
      if (c + 1 < chunks) {
        chunk(c + 1, wb, wa);
      } else {
#pragma unroll
        for (int j = 0; j < TN; ++j) wa[j] = wb[j];
      }
    }
    if (GLU) {
      // (the sums made again in one place, for each of the 64: written out for each they cost 4 us a tile in code alone)
      const int c = n0 + 16 * wave + 4 * lg;     // (N is a multiple of 4)
      unsigned odd[2] = {0, 0};
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int m = m0 + 16 * i + ln;
        if (m >= M || c >= N) continue;
        f32x4_t out;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          out[e] = glu_act(a.act, sum[0][i][e]) * sum[TN - 1][i][e];
          odd[0] |= is_finite(sum[0][i][e]) ? 0u : 1u << (4 * i + e);
          odd[1] |= is_finite(sum[TN - 1][i][e]) ? 0u : 1u << (4 * i + e);
        }
        *reinterpret_cast<f32x4_t*>(a.y + (size_t)m * a.ldy + c) = out;
      }
      if (__builtin_expect(__any(odd[0] | odd[1]), 0)) {
        bool nan_x = false;
#pragma unroll 1
        for (int k = 0; k < 4 * TM; ++k) {
          if (k % 4 == 0) nan_x = false;         // (other rows of x)
          const bool again = (odd[0] | odd[1]) >> k & 1;
          if (!__any(again)) continue;
          const size_t m = min(m0 + 16 * (k >> 2) + ln, M - 1), col = min(c, N - 4) + (k & 3);
          float g = 0.f, u = 0.f;
#pragma unroll
          for (int q = 0; q < 4 * TM; ++q) {
            g = q == k ? sum[0][q >> 2][q & 3] : g;
            u = q == k ? sum[TN - 1][q >> 2][q & 3] : u;
          }
#pragma unroll 1
          for (int side = 0; side < 2; ++side) {
            const float v = plain_dots(side ? u : g, odd[side] >> k & 1, a.x + m * a.ldx,
                                       a.w + (side * (size_t)N + col) * K, K, nan_x);
            if (side) u = v; else g = v;
          }
          if (again) a.y[m * a.ldy + col] = glu_act(a.act, g) * u;
        }
      }
    } else if (!PARTS) {
      tile_again<4 * TN, TM>(a.y, a.ldy, store(a.y, a.ldy, sum), m0, n0 + 16 * TN * wave, M, N, a.x, a.ldx, a.w, K);
    }
  }
}

// The tiles there are: rows of x and of W, buffers, workgroups a compute unit, and what one takes, in us: R rounds of
// workgroups with c blocks of 32 columns each, of which a share f of the chip's places is taken, take
// R (c (block + full f) + 2). The last one is gemm_f32_tile_kernel's.
#define STREAM_TILES(T)                       \
  T(128, 128, 4, 1, 0.98f, 0.27f)             \
  T(64, 128, 5, 1, 0.65f, 0.08f)              \
  T(64, 64, 4, 2, 0.44f, 0.33f)
constexpr int LOADERS = 4;

constexpr int N_STREAMS = 3;

struct TilePlan {
  int tile;                                      // of STREAM_TILES, or N_STREAMS: gemm_f32_tile_kernel
  int bm, bn;                                    // rows of x and of W a tile
  int per;                                       // columns a workgroup
  int per_cu;
  float us;
};

// pairs: W is [Wg; Wu] and the pairs are finished in the tile, for which K is not cut
static TilePlan tile_plan(int M, int N, int K, bool pairs = false) {
  const int cus = compute_units();
  const int width = span_width(K), spans = (K + width - 1) / width;
  TilePlan best{};
  double least = 1e30;
  auto offer = [&](int tile, int bm, int bn, int per_cu, float block, float full) {
    const long tiles = (long)((N + bn - 1) / bn) * ((M + bm - 1) / bm);
    if (pairs && bn != 128) return;
    for (int splits = 1; splits <= (pairs ? 1 : spans); ++splits) {
      const int per = (spans + splits - 1) / splits * width;
      if ((long)per * (splits - 1) >= K) continue;
      const long places = (long)cus * per_cu, all = tiles * splits, rounds = (all + places - 1) / places;
      const double c = (min(per, K) + SPLIT_BK - 1) / SPLIT_BK;
      double t = rounds * (c * (block + full * (double)all / (rounds * places)) + 2.0);
      if (splits > 1) t += 4.0 + 4.0 * M * N * (spans + 1) / 6e6;
      if (t < least) {
        least = t;
        best = {tile, bm, bn, per, per_cu, (float)t};
      }
    }
  };
  if (K % SPLIT_BK == 0) {
    int n = 0;
#define T(BM, BN, NB, CU, BLOCK, FULL) offer(n++, BM, BN, CU, BLOCK, FULL);
    STREAM_TILES(T)
#undef T
    // Spans of four blocks and a grid that lies on the chip at once with one span a workgroup: there the kernel that splits x
    // costs more than its parts save (one MI355X, us, this form against the best of the others: 300 x 200 x 96 5.8 / 7.1, 17 x 256 x
    // 512 8.1 / 9.0, 300 x 512 x 512 9.4 / 10.9, 128 x 1,024 x 1,024 10.9 / 12.3, 100 x 3,072 x 768 16.1 / 16.3, 130 x 16,384 x 128
    // 11.8 / 13.9). Not with more of it, 130 x 4,096 x 512 17.2 / 13.3, 64 x 7,000 x 1,024 22.4 / 20.8, 700 x 16,384 x 128 32 / 29,
    // and not with longer spans, where neither is ahead, 17 x 2,048 x 2,048 13.3 / 12.9, 64 x 3,072 x 2,048 17.5 / 18.8.
    const long tiles = (long)((N + 63) / 64) * ((M + 63) / 64);
    if (!pairs && width == 128 && 2 * tiles * spans <= (spans > 1 ? 5L : 8L) * cus)
      best = {N_STREAMS, 64, 64, width, 4, best.us - 1.5f};
  } else {
    offer(N_STREAMS, 64, 64, 4, 1.3f, 0.35f);
  }
  return best;
}

static int padded_rows(int M) { return (M + 127) / 128 * 128; }

// floats of the parts of x
static long split_rows_floats(const TilePlan& plan, int M, int K) {
  return plan.tile == N_STREAMS ? 0 : (long)(split_rows_bytes(padded_rows(M)) / 4) * (K / SPLIT_BK);
}

template <int BM, int BN, int NB, int MODE> static int launch_stream(const StreamArgs& a, int per_cu, hipStream_t st) {
  constexpr size_t lds = (size_t)NB * (BN + BM + BM / 2) * TILE_ROW;
  static LdsAllowance allowance;
  if (!allowance.ask((const void*)gemm_f32_stream_kernel<BM, BN, NB, LOADERS, MODE>, lds)) return PTL_ERR_LAUNCH;
  const long tiles = (long)a.tiles_m * a.tiles_n * a.splits;
  const unsigned grid = (unsigned)min(tiles, (long)compute_units() * per_cu);
  gemm_f32_stream_kernel<BM, BN, NB, LOADERS, MODE><<<grid, 64 * (4 + LOADERS), lds, st>>>(a);
  return ptl_launch_status();
}

// work: split_rows_floats, then the spans' sums if K is cut
static int launch_tiles(float* y, const float* x, const float* w, int M, int N, int K, long ldx, long ldy,
                        const TilePlan& plan, float* work, hipStream_t st) {
  const int width = span_width(K), spans = (K + width - 1) / width;
  const int tiles_m = (M + plan.bm - 1) / plan.bm, tiles_n = (N + plan.bn - 1) / plan.bn;
  const int splits = (K + plan.per - 1) / plan.per;
  if ((long)tiles_m * tiles_n * splits > 0x3fffffff) return PTL_ERR_ARG;
  float* parts = splits > 1 ? work + split_rows_floats(plan, M, K) : nullptr;
  if (plan.tile == N_STREAMS) {
    const long tiles = (long)tiles_m * tiles_n;
    const dim3 grid((unsigned)((tiles + 7) / 8 * 8), splits);
    (parts ? gemm_f32_tile_kernel<1, 4, true> : gemm_f32_tile_kernel<1, 4, false>)<<<grid, 256, 0, st>>>(
        y, x, w, M, N, K, ldx, ldy, tiles_m, (int)tiles, width, plan.per, parts);
  } else {
    const int Mp = padded_rows(M);
    unsigned char* xs = reinterpret_cast<unsigned char*>(work);
    split_rows_kernel<<<dim3((M + 63) / 64, K / SPLIT_BK), 256, 0, st>>>(xs, x, M, K, ldx, Mp);
    const StreamArgs a{y, parts, x, w, xs, M, N, K, Mp, ldx, ldy, tiles_m, tiles_n, splits, plan.per, width, 0};
    int rc = PTL_ERR_ARG, n = 0;
#define T(BM, BN, NB, CU, BLOCK, FULL)                                                                   \
  if (plan.tile == n++)                                                                                  \
    rc = parts ? launch_stream<BM, BN, NB, STREAM_PARTS>(a, CU, st) : launch_stream<BM, BN, NB, STREAM_Y>(a, CU, st);
    STREAM_TILES(T)
#undef T
    if (rc != PTL_OK) return rc;
  }
  if (parts)
    gemm_f32_sum_kernel<<<(unsigned)(((long)M * N + 1023) / 1024), 256, 0, st>>>(y, parts, spans, x, w, M, N, K, ldx, ldy);
  return ptl_launch_status();
}

static long workspace_floats(const TilePlan& plan, int M, int N, int K) {
  const int width = span_width(K);
  return split_rows_floats(plan, M, K) + (plan.per < K ? (long)((K + width - 1) / width) * M * N : 0);
}

// floats of workspace ptl_gemm_f32 wants for these sizes (0: none)
extern "C" long ptl_gemm_f32_workspace(int M, int N, int K) {
  return M <= 0 || N <= 0 || K <= 0 ? 0 : workspace_floats(tile_plan(M, N, K), M, N, K);
}

// K % 4 == 0, ldx % 4 == 0, x and w 16-byte aligned. ``work``: workspace of ptl_gemm_f32_workspace(M, N, K)
// floats, 16-byte aligned (null where that is 0).
extern "C" int ptl_gemm_f32(float* y, const float* x, const float* w, int M, int N, int K, long ldx, long ldy,
                            float* work, hipStream_t st) {
  if (M <= 0 || N <= 0) return PTL_OK;
  if (K <= 0 || K % 4 || (M > 1 && ldx % 4) || ldx < K || ldy < N || !aligned16(x) || !aligned16(w)) return PTL_ERR_ARG;
  const TilePlan plan = tile_plan(M, N, K);
  if (workspace_floats(plan, M, N, K) > 0 && (work == nullptr || !aligned16(work))) return PTL_ERR_ARG;
  return launch_tiles(y, x, w, M, N, K, ldx, ldy, plan, work, st);
}

// The plan with tile number ``tile`` and the spans in ``splits`` parts; false if there is none.
static bool plan_with(int M, int N, int K, int tile, int splits, TilePlan& plan) {
  const int width = span_width(K), spans = (K + width - 1) / width;
  if (M <= 0 || N <= 0 || K <= 0 || K % 4 || splits < 1 || splits > spans || tile < 0 || tile > N_STREAMS ||
      (tile < N_STREAMS && K % SPLIT_BK))
    return false;
  static const int sizes[][3] = {
#define T(BM, BN, NB, CU, BLOCK, FULL) {BM, BN, CU},
      STREAM_TILES(T)
#undef T
      {64, 64, 4}};
  static_assert(sizeof(sizes) / sizeof(sizes[0]) == N_STREAMS + 1, "");
  const int per = (spans + splits - 1) / splits * width;
  if ((long)per * (splits - 1) >= K) return false;
  plan = {tile, sizes[tile][0], sizes[tile][1], per, sizes[tile][2], 0.f};
  return true;
}

// ptl_gemm_f32 by a tile of its own choice, and what it wants (-1: there is no such plan)
extern "C" long ptl_gemm_f32_tiles_workspace(int M, int N, int K, int tile, int splits) {
  TilePlan plan;
  return plan_with(M, N, K, tile, splits, plan) ? workspace_floats(plan, M, N, K) : -1;
}

extern "C" int ptl_gemm_f32_tiles(float* y, const float* x, const float* w, int M, int N, int K, long ldx, long ldy, int tile,
                                  int splits, float* work, hipStream_t st) {
  TilePlan plan;
  if (!plan_with(M, N, K, tile, splits, plan) || (M > 1 && ldx % 4) || ldx < K || ldy < N || !aligned16(x) || !aligned16(w) ||
      (workspace_floats(plan, M, N, K) > 0 && (work == nullptr || !aligned16(work))))
    return PTL_ERR_ARG;
  return launch_tiles(y, x, w, M, N, K, ldx, ldy, plan, work, st);
}

// Whether ptl_gate_up_f32_tiles is the faster way for M rows of x and W = [Wg; Wu] [2 I, K]: what the plans say, the activation's
// kernel taking 3 us and its 12 bytes a result at 5 TB/s (700 rows, 2 x 8,192 x 2,048: 15 to 16 us).
extern "C" int ptl_gate_up_f32_tiles_fits(int M, int I, int K) {
  if (M <= 0 || I <= 0 || I % 4 || K <= 0 || K % SPLIT_BK) return 0;
  return tile_plan(M, 2 * I, K, true).us <= tile_plan(M, 2 * I, K).us + 3.0f + 12.0f * M * I / 5e6f;
}

// floats of workspace it wants
extern "C" long ptl_gate_up_f32_tiles_workspace(int M, int I, int K) {
  return M <= 0 || I <= 0 || K <= 0 ? 0 : split_rows_floats(tile_plan(M, 2 * I, K, true), M, K);
}

// out [M, I] = act(x Wg^T) * (x Wu^T), the bits of the product and the activation by themselves. K % 32 == 0, I % 4 == 0, ldx % 4
// == 0, 16-byte aligned rows and workspace.
extern "C" int ptl_gate_up_f32_tiles(float* out, const float* x, const float* w, int M, int I, int K, long ldx, int act,
                                     float* work, hipStream_t st) {
  if (M <= 0) return PTL_OK;
  if (I <= 0 || I % 4 || K <= 0 || K % SPLIT_BK || (M > 1 && ldx % 4) || ldx < K || !aligned16(out) || !aligned16(x) ||
      !aligned16(w) || !work || !aligned16(work) || (act != GLU_SILU && act != GLU_GELU_TANH))
    return PTL_ERR_ARG;
  const TilePlan plan = tile_plan(M, 2 * I, K, true);
  const int tiles_m = (M + plan.bm - 1) / plan.bm, tiles_n = (I + 63) / 64, Mp = padded_rows(M);
  if ((long)tiles_m * tiles_n > 0x3fffffff) return PTL_ERR_ARG;
  unsigned char* xs = reinterpret_cast<unsigned char*>(work);
  split_rows_kernel<<<dim3((M + 63) / 64, K / SPLIT_BK), 256, 0, st>>>(xs, x, M, K, ldx, Mp);
  const StreamArgs a{out, nullptr, x, w, xs, M, I, K, Mp, ldx, I, tiles_m, tiles_n, 1, K, span_width(K), act};
  if (plan.bm == 128) return launch_stream<128, 128, 4, STREAM_GLU>(a, 1, st);
  return launch_stream<64, 128, 5, STREAM_GLU>(a, 1, st);
}
