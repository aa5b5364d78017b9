// y = x W^T in float32 on the matrix cores: row-major x [M, K] (row stride ldx) and W [N, K],
// float32 products and sums (v_mfma_f32_16x16x4_f32 multiplies and adds in float32, so this is the same
// true 32-bit arithmetic as the vector-FMA kernel of gemm.hip, in another order).
//
// All kernels need K % 4 == 0 and 16-byte aligned rows of x and W; everything else stays with the
// vector-FMA kernel.
//
// One order of sums. The bits of a result do not depend on the other rows of x, nor on how many there are, so
// that a request's float32 results are the same alone and in a batch: all kernels add the products of a result
// in an order that K alone fixes. The columns are cut into spans of span_width(K) (at most 16). A span's sum is
// that of its even plus that of its odd blocks of 16 columns; either starts from zero and takes its blocks one
// after the other, four matrix instructions a block, of which number s multiplies columns 3 - s, 7 - s, 11 - s and
// 15 - s (a lane loads four consecutive columns at once and hands them to the four instructions). The spans'
// sums are added in order. Which wave, workgroup or lane computes a span is free. (Measured, in us, against
// kernels whose order followed M: level at up to 8 rows; 64 x 2,048 x 2,048 19.0 -> 15.0, 700 x 2,048 x 2,048 76 -> 80,
// 300 x 4,096 x 4,096 116 -> 128, 17 x 16 x 2,048 8.9 -> 10.9; a prompt of 700 tokens and a decode step of four rows at
// the Llama-3.2-1B shape are level, their errors against 64 bits 1.1e-6 -> 4.1e-7 and 4.5e-7 -> 3.9e-7.)
#include "common.h"
#include "device.h"
#include "mfma_f32.h"

// columns of a span: 256, doubled until there are no more than 16; 128 of short sums, which have few spans to share
__host__ __device__ static inline int span_width(int K) {
  int w = K <= 1024 ? 128 : 256;
  while ((long)w * 16 < K) w <<= 1;
  return w;
}

// ===========================================================================
// Few rows of x (M <= 16, a decode step): bound by reading W once. A workgroup owns ROWS rows of W;
// its waves take the spans, every wave keeps up to 16 KB of W under way (two sets of U
// loads of 1 KB), and the spans' sums meet in LDS. v_mfma_f32_16x16x4_f32: lane l (ln = l % 16,
// lg = l / 16) holds A[ln][k = lg] and B[k = lg][ln] and gets D[4 lg + i][ln].
//
// ROWS 16: A is 16 rows of W x 16 columns, a load instruction reads 64 bytes of each row; B the same
// columns of 16 rows of x, from L2. Even and odd blocks have sums of their own.
// ROWS 8: with at most 8 rows of x half of such a tile would be empty, so the tile holds two blocks of
// 16 columns of the same 8 rows (lanes ln < 8 the even block, ln >= 8 the odd one), of W and of x
// alike. The products that matter are then D[n < 8][m < 8] and D[n >= 8][m >= 8], the sums of the even and
// of the odd blocks, and every load instruction, of W and of x, still brings 1 KB that is used. It gives twice
// the workgroups. MT tiles of 8 rows of x share the loads of W.
//
// gemm_f32_few_kernel reads x again for every tile and takes the sums of any length;
// gemm_f32_held_kernel keeps x in registers and walks several tiles.
//
// Measured (one MI355X, cold weights, us at 4 rows; in brackets the vector-FMA kernel that ran first and
// gemm_f32_few_kernel): 16,384 x 2,048 26 = 5.2 TB/s (240, 33), 2,048 x 8,192 17 = 4.0 TB/s (922, 18.5),
// 128,256 x 2,048 171 = 6.1 TB/s (643, 214), 2,048 x 2,048 6.7 (209), 64 x 256 3.6 (25); a decode step of 4 rows at
// the Llama-3.2-1B shape 1.57 ms (28.2).
// ===========================================================================

// A tile's results from the spans' sums in LDS ([span][MT][64 lanes][4], lane and element as in D; of 8-row tiles
// the two halves).
template <int ROWS, int MT>
__device__ __forceinline__ void few_results(float* __restrict__ y, const float* sums, int spans, int M, int N, int n0,
                                            long ldy) {
  for (int i = threadIdx.x; i < ROWS * ROWS * MT; i += blockDim.x) {
    const int n = i % ROWS, m = i / ROWS, t = m / ROWS, j = m % ROWS;
    if (m >= M || n0 + n >= N) continue;
    const float* p = sums + t * 256 + ((n >> 2) * 16 + j) * 4 + (n & 3);
    constexpr int ODD = (2 * 16 + 8) * 4;          // from D[n][j] to D[n + 8][j + 8]
    float s = 0.f;
    for (int sp = 0; sp < spans; ++sp, p += MT * 256) s += ROWS == 8 ? p[0] + p[ODD] : p[0];
    y[(size_t)m * ldy + n0 + n] = s;
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
__device__ __forceinline__ void pair_results(float* __restrict__ y, const float* sums, int spans, int M, int tile, long ldy,
                                             const FewOut& o) {
  for (int i = threadIdx.x; i < 32; i += blockDim.x) {
    const int n = i & 3, m = i >> 2;
    if (m >= M) continue;
    const float *p = sums + m * 4 + n, *p2 = p + 16 * 4;
    constexpr int ODD = (2 * 16 + 8) * 4;
    float a = 0.f, b = 0.f;
    for (int sp = 0; sp < spans; ++sp, p += 256, p2 += 256) {
      a += p[0] + p[ODD];
      b += p2[0] + p2[ODD];
    }
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

template <int ROWS, int MT, int U>
__global__ void __launch_bounds__(1024)
gemm_f32_few_kernel(float* __restrict__ y, const float* __restrict__ x, const float* __restrict__ w,
                    int M, int N, int K, long ldx, long ldy, int width) {
  extern __shared__ float red[];                 // [waves][MT][64][4]: a wave a span
  static_assert((ROWS == 16 && MT == 1) || ROWS == 8, "rows of W a tile");
  constexpr int KB = ROWS == 8 ? 32 : 16;        // columns of W that one load instruction covers
  constexpr int H = ROWS == 8 ? 1 : 2;           // sums a lane keeps of a tile
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, ln = lane & 15, lg = lane >> 4;
  const int n0 = blockIdx.x * ROWS;
  const int koff = 4 * lg + (ROWS == 8 ? 16 * (ln >> 3) : 0);
  const float* wp = w + (size_t)min(n0 + ln % ROWS, N - 1) * K + koff;
  const float* xp[MT];
  bool xok[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = ROWS * t + ln % ROWS;
    xok[t] = m < M;
    xp[t] = x + (size_t)min(m, M - 1) * ldx + koff;
  }
  f32x4_t acc[MT][H];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int h = 0; h < H; ++h) acc[t][h] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int kb = wave * width;
  const int ke = min(K, kb + width);
  // two sets of weight registers: the next U blocks are under way while these are multiplied
  F4 wa[U], wb[U];
  auto load_w = [&](F4 (&f)[U], int k) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool ok = k + KB * u + koff < ke;
      f[u].u = ok ? load_once(wp + k + KB * u) : zero16();
    }
  };
  auto multiply = [&](const F4 (&f)[U], int k) {
    F4 xf[MT][U];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const bool ok = xok[t] && k + KB * u + koff < ke;
        xf[t][u].u = ok ? load16(xp[t] + k + KB * u) : zero16();
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          acc[t][u % H] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[u].f[3 - s], xf[t][u].f[3 - s], acc[t][u % H], 0, 0, 0);
  };
  if (kb < ke) load_w(wa, kb);
  for (int k = kb; k < ke; k += 2 * KB * U) {
    const int k1 = k + KB * U, k2 = k + 2 * KB * U;
    if (k1 < ke) load_w(wb, k1);
    multiply(wa, k);
    if (k1 >= ke) break;
    if (k2 < ke) load_w(wa, k2);
    multiply(wb, k1);
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    f32x4_t s = acc[t][0];
    if (H == 2)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] += acc[t][H - 1][i];
    *reinterpret_cast<f32x4_t*>(red + (((size_t)wave * MT + t) * 64 + lane) * 4) = s;
  }
  __syncthreads();
  few_results<ROWS, MT>(y, red, blockDim.x >> 6, M, N, n0, ldy);
}

// Up to 8 rows (16 of 16-row tiles) with a wave's share of the columns in registers: x [ROWS, KB NB] of every wave
// is read once, and the workgroup then walks ROWS-row tiles of W (blockIdx.x, + gridDim.x, ...), so that W is all that
// is read in the loop: read again for every tile, x comes through the same path from L2 as W does and is as many
// bytes (128,256 x 2,048, us at 1, 4 and 8 rows: 185, 214, 254; held 161, 171, 177). The next tile's first columns are on their way while a tile's
// sums are added up, in two buffers, one barrier a tile. SB: load blocks of a span.
template <int ROWS, int NB, int SB, int FORM>
__global__ void __launch_bounds__(1024)
gemm_f32_held_kernel(float* __restrict__ y, const float* __restrict__ x, const float* __restrict__ w,
                     int M, int N, int K, long ldx, long ldy, int tiles, FewOut out) {
  static_assert(ROWS == 8 || FORM == FORM_PLAIN, "pairs lie in 8-row tiles");
  constexpr int KB = ROWS == 8 ? 32 : 16;        // columns of a block (as above)
  constexpr int H = ROWS == 8 ? 1 : 2;
  constexpr int U = 4, S = NB / U;               // blocks a turn, turns a tile
  constexpr int EACH = NB / SB;                  // spans of a wave
  static_assert(S % 2 == 0, "the two sets of registers change places an even number of times a tile");
  static_assert(NB % SB == 0 && SB % U == 0, "a turn does not cross a span's end, a wave's share ends with a span");
  extern __shared__ float red[];                 // [2][waves][EACH][64][4]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, ln = lane & 15, lg = lane >> 4;
  const int nwaves = blockDim.x >> 6;
  const int kb = KB * NB * wave + 4 * lg + (ROWS == 8 ? 16 * (ln >> 3) : 0);
  const int left = K - kb;                       // this lane's columns of block b are there if KB b < left
  F4 xf[NB];
  {
    const float* xp = x + (size_t)min(ln % ROWS, M - 1) * ldx + kb;
    const bool row = ln % ROWS < M;
#pragma unroll
    for (int b = 0; b < NB; ++b) xf[b].u = row && KB * b < left ? load16(xp + KB * b) : zero16();
  }
  F4 wa[U], wb[U];
  auto load_w = [&](F4 (&f)[U], int tile, int b0) __attribute__((always_inline)) {
    const float* wp = w + (size_t)few_row<FORM, ROWS>(out, tile, ln % ROWS, N) * K + kb;
#pragma unroll
    for (int u = 0; u < U; ++u) f[u].u = KB * (b0 + u) < left ? load_once(wp + KB * (b0 + u)) : zero16();
  };
  load_w(wa, blockIdx.x, 0);
  int at = 0;
  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x, at ^= 1) {
    float* const sums = red + at * nwaves * EACH * 256;
    f32x4_t acc[H];
#pragma unroll
    for (int h = 0; h < H; ++h) acc[h] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < S; ++s) {
      F4 (&cur)[U] = s % 2 ? wb : wa;
      F4 (&next)[U] = s % 2 ? wa : wb;
      if (s + 1 < S) load_w(next, tile, U * (s + 1));
      else if (tile + (int)gridDim.x < tiles) load_w(next, tile + gridDim.x, 0);
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc[u % H] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur[u].f[3 - i], xf[U * s + u].f[3 - i], acc[u % H], 0, 0, 0);
      if ((s + 1) * U % SB == 0) {               // the end of a span
        if (H == 2)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[0][i] += acc[H - 1][i];
        *reinterpret_cast<f32x4_t*>(sums + ((wave * EACH + s * U / SB) * 64 + lane) * 4) = acc[0];
#pragma unroll
        for (int h = 0; h < H; ++h) acc[h] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    }
    __syncthreads();
    if (FORM == FORM_PLAIN) few_results<ROWS, 1>(y, sums, nwaves * EACH, M, N, ROWS * tile, ldy);
    else pair_results<FORM>(y, sums, nwaves * EACH, M, tile, ldy, out);
  }
}

// x in registers, tiles of ``rows`` rows of W: up to 8 rows of x and 8,192 columns, or 16 and 4,096.
template <int FORM>
static int launch_held(float* y, const float* x, const float* w, int M, int N, int K, long ldx, long ldy, int rows,
                       const FewOut& out, hipStream_t st) {
  const int cus = compute_units();
  const long blocks = (N + rows - 1) / rows;
  const int width = span_width(K);
  // (8 rows: 512 columns a wave where that gives 64 waves a compute unit, else 256)
  const bool half = rows == 8 && K <= 4096 && blocks * ((K + 511) / 512) < 64L * cus;
  const int share = rows == 8 && !half ? 512 : 256;
  const int waves = (K + share - 1) / share;
  const long resident = (long)cus * (16 / waves);
  const long walk = (blocks + resident - 1) / resident;
  const unsigned grid = (unsigned)((blocks + walk - 1) / walk);
#define HELD(ROWS, NB, SB)                                                                                      \
  gemm_f32_held_kernel<ROWS, NB, SB, ROWS == 8 ? FORM : FORM_PLAIN>                                             \
      <<<grid, waves * 64, (size_t)waves * (NB / SB) * 2048, st>>>(y, x, w, M, N, K, ldx, ldy, (int)blocks, out)
  if (rows == 16 && width == 128) HELD(16, 16, 8);
  else if (rows == 16) HELD(16, 16, 16);
  else if (half && width == 128) HELD(8, 8, 4);
  else if (half) HELD(8, 8, 8);
  else if (width == 128) HELD(8, 16, 4);
  else if (width == 256) HELD(8, 16, 8);
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
  const long blocks = (N + rows - 1) / rows;
  const int width = span_width(K), spans = (K + width - 1) / width;
  // x in registers where it fits, up to 512 columns a wave of 8 rows or 256 of 16, 16 waves a compute unit
  // (16 rows, read again against held: 16,384 x 2,048 43 / 36, 3,072 x 2,048 12.0 / 12.2, 128,256 x 2,048 317 / 230;
  // not where 8-row tiles are taken for more than 8 rows: 2,048 x 2,048 10.4 / 11.3)
  if (rows == 8 ? M <= 8 && K <= 8192 : K <= 4096) {
    return launch_held<FORM_PLAIN>(y, x, w, M, N, K, ldx, ldy, rows, FewOut{}, st);
  }
#define GO(ROWS, MT)                                                                                        \
  gemm_f32_few_kernel<ROWS, MT, 8 / MT><<<(unsigned)blocks, spans * 64, (size_t)spans * MT * 1024, st>>>(y, x, w, M, N, K, \
                                                                                                       ldx, ldy, width)
  if (rows == 16) GO(16, 1);
  else if (M <= 8) GO(8, 1);
  else GO(8, 2);
#undef GO
  return ptl_launch_status();
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
  return launch_held<FORM_GLU>(out, x, w, M, 2 * I, K, ldx, I, 8, o, st);
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
  return launch_held<FORM_QKV>(q_out, x, w, M, (Hq + 2 * Hkv) * D, K, ldx, (long)Hq * D, 8,
                               FewOut{D / 2, 0, positions, slots, inv_freq, k_cache, v_cache, Hq, Hkv, page_size}, st);
}

// ===========================================================================
// Many rows of x (a prompt portion): tiles of 64 rows of W x 64 rows of x a workgroup of four waves, each 32 x 32,
// F32_BK columns of K at a time through LDS, two buffers: the next tile is on its way from memory to registers
// while this one is multiplied, one barrier a tile. For 16 columns a wave reads four 16-byte fragments a lane and
// issues 16 matrix instructions of 32 clocks each (mfma_f32.h), so the matrix cores bound it. A wave keeps its
// results three times, the sums of the even blocks, of the odd blocks and of the spans so far; at the end of a
// span the first two are added to the third. (Tiles of 128 x 64 and 128 x 128, M 17 to 2,048, N 1,536 to 28,672: at
// most 5 % faster anywhere, up to 40 % slower.)
//
// A grid of few tiles is cut along K as well (blockIdx.y, a number of spans each): the spans' sums go to a
// workspace [spans, M, N] and a second kernel adds them in order.
//
// Measured (one MI355X, us; the vector-FMA kernel that ran before in brackets): 700 x 16,384 x 2,048 432 =
// 109 TFLOP/s (1,386), 700 x 2,048 x 8,192 237 (1,251), 700 x 3,072 x 2,048 115 (370), 64 x 2,048 x 8,192 30.5 (963),
// 17 x 2,048 x 2,048 13.5 (228). Relative error against 64 bits of a 700-token prompt's logits at the Llama-3.2-1B shape
// 4.1e-7 (1.5e-6).
// ===========================================================================
#define F32_TILE 64
// (two workgroups a unit asked for: without it the sums go to accumulation registers and the occupancy falls)
__global__ void __launch_bounds__(256, 2)
gemm_f32_tile_kernel(float* __restrict__ y, const float* __restrict__ x, const float* __restrict__ w,
                     int M, int N, int K, long ldx, long ldy, int tiles_m, int tiles, int width, int k_per_split,
                     float* __restrict__ parts) {
  constexpr int T = 2;                           // 16 x 16 results of a wave along each side
  constexpr int L = F32_TILE / 32;               // 16-byte pieces of W and of x a thread loads, of rows 32 apart
  __shared__ uint4 ws[2][F32_TILE * 8];
  __shared__ uint4 xs[2][F32_TILE * 8];
  // Workgroups go to the eight XCDs in turn: each gets a run of tiles, neighbours in the run share
  // rows of W, so that W comes into one L2 once.
  const int per_xcd = (tiles + 7) / 8;
  const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (tile >= tiles || (int)(blockIdx.x >> 3) >= per_xcd) return;
  const int n0 = tile / tiles_m * F32_TILE, m0 = tile % tiles_m * F32_TILE;
  const int kb = blockIdx.y * k_per_split, ke = min(K, kb + k_per_split);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, ln = lane & 15, lg = lane >> 4;
  const int wn = 32 * (wave & 1), wm = 32 * (wave >> 1);
  const int piece = tid & 7, row = tid >> 3;
  const float* wp[L];
  const float* xp[L];
#pragma unroll
  for (int i = 0; i < L; ++i) wp[i] = w + (size_t)min(n0 + row + 32 * i, N - 1) * K + 4 * piece;
#pragma unroll
  for (int i = 0; i < L; ++i) xp[i] = x + (size_t)min(m0 + row + 32 * i, M - 1) * ldx + 4 * piece;
  uint4 wr[L], xr[L];
  auto fetch = [&](int k) {
    const bool ok = k + 4 * piece < ke;
#pragma unroll
    for (int i = 0; i < L; ++i) wr[i] = ok ? load16(wp[i] + k) : zero16();
#pragma unroll
    for (int i = 0; i < L; ++i) xr[i] = ok ? load16(xp[i] + k) : zero16();
  };
  auto put = [&](int b) {
#pragma unroll
    for (int i = 0; i < L; ++i) ws[b][f32_piece(row + 32 * i, piece)] = wr[i];
#pragma unroll
    for (int i = 0; i < L; ++i) xs[b][f32_piece(row + 32 * i, piece)] = xr[i];
  };
  // results [M, N] of row stride ld, from D[n = 4 lg + i][m = ln] of every 16 x 16 tile
  auto store = [&](float* to, long ld, const f32x4_t (&v)[T][T]) {
    const bool four = (N & 3) == 0 && (ld & 3) == 0 && (reinterpret_cast<uintptr_t>(to) & 15) == 0;
#pragma unroll
    for (int c = 0; c < T; ++c) {
      const int m = m0 + wm + 16 * c + ln;
      if (m >= M) continue;
#pragma unroll
      for (int a = 0; a < T; ++a) {
        const int n = n0 + wn + 16 * a + 4 * lg;
        float* at = to + (size_t)m * ld + n;
        if (four) {
          if (n < N) *reinterpret_cast<f32x4_t*>(at) = v[a][c];
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (n + i < N) at[i] = v[a][c][i];
        }
      }
    }
  };
  f32x4_t acc[2][T][T], sum[T][T];           // acc: of the span's even and of its odd blocks
#pragma unroll
  for (int a = 0; a < T; ++a)
#pragma unroll
    for (int c = 0; c < T; ++c) acc[0][a][c] = acc[1][a][c] = sum[a][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  fetch(kb);
  put(0);
  __syncthreads();
  int buf = 0;
  for (int k = kb; k < ke; k += F32_BK, buf ^= 1) {
    const bool more = k + F32_BK < ke;
    if (more) fetch(k + F32_BK);
    f32_multiply16<T, T>(acc, ws[buf], xs[buf], wn, wm, lane);
    if (!more || (k + F32_BK) % width == 0) {    // the end of a span
#pragma unroll
      for (int a = 0; a < T; ++a)
#pragma unroll
        for (int c = 0; c < T; ++c) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float s = acc[0][a][c][i] + acc[1][a][c][i];
            sum[a][c][i] = parts ? s : sum[a][c][i] + s;
          }
          acc[0][a][c] = acc[1][a][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
      if (parts) store(parts + (size_t)(k / width) * M * N, N, sum);
    }
    if (more) put(buf ^ 1);
    __syncthreads();
  }
  if (!parts) store(y, ldy, sum);
}

__global__ void __launch_bounds__(256)
gemm_f32_sum_kernel(float* __restrict__ y, const float* __restrict__ parts, int spans, int M, int N, long ldy) {
  const long total = (long)M * N;
  if ((N & 3) == 0 && (ldy & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0) {
    const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= total) return;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
    for (int p = 0; p < spans; ++p) {
      const float4 v = *reinterpret_cast<const float4*>(parts + (size_t)p * total + i);
      s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
    *reinterpret_cast<float4*>(y + i / N * ldy + i % N) = s;
    return;
  }
  for (int j = 0; j < 4; ++j) {
    const long i = (long)blockIdx.x * 1024 + j * 256 + threadIdx.x;
    if (i >= total) return;
    float s = 0.f;
    for (int p = 0; p < spans; ++p) s += parts[(size_t)p * total + i];
    y[i / N * ldy + i % N] = s;
  }
}

// Columns that a workgroup takes (a number of spans; all: no second kernel): what a count of the work says is done
// first. The waves of a workgroup take the four SIMDs of a compute unit, so what counts is the fullest unit: r
// workgroups, one after the other, at 0.5 TFLOP/s (128 TFLOP/s on 256 units), each with about two
// steps of F32_BK lost at its start and end; less than three at a time on a unit leave gaps (one alone
// takes 1.6 times as long). Cuts cost the second kernel and the traffic of the spans' sums, however many they are.
// Against a sweep of all numbers of cuts (M 17 to 700, N 16 to 28,672, K 512 to 14,336; one MI355X) the plan is
// within 6 % of the fastest; without cuts 64 x 2,048 x 8,192 takes 140 instead of 31.
static int columns_a_split(int M, int N, int K) {
  const int cus = compute_units();
  const int width = span_width(K), spans = (K + width - 1) / width;
  const long tiles = (long)((N + F32_TILE - 1) / F32_TILE) * ((M + F32_TILE - 1) / F32_TILE);
  int best = spans * width;
  double least = 1e30;
  for (int splits = 1; splits <= spans; ++splits) {
    const int per = (spans + splits - 1) / splits * width;
    if ((long)per * (splits - 1) >= K) continue;
    const double one = 2.0 * F32_TILE * F32_TILE * (min(per, K) + 2 * F32_BK) / 0.5e12;
    const double r = (double)((tiles * splits + cus - 1) / cus);
    double t = one * (r < 4 ? 0.8 * (r + 1) : r + 0.3);
    if (splits > 1) t += 4e-6 + 4.0 * M * N * (spans + 1) / 6e12;
    if (t < least) {
      least = t;
      best = per;
    }
  }
  return best;
}

// floats of workspace ptl_gemm_f32 wants for these sizes (0: none)
extern "C" long ptl_gemm_f32_workspace(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const int width = span_width(K);
  return columns_a_split(M, N, K) < K ? (long)((K + width - 1) / width) * M * N : 0;
}

// K % 4 == 0, ldx % 4 == 0, x and w 16-byte aligned. ``parts``: workspace of ptl_gemm_f32_workspace(M, N, K)
// floats, 16-byte aligned (null where that is 0).
extern "C" int ptl_gemm_f32(float* y, const float* x, const float* w, int M, int N, int K, long ldx, long ldy,
                            float* parts, hipStream_t st) {
  if (M <= 0 || N <= 0) return PTL_OK;
  if (K <= 0 || K % 4 || (M > 1 && ldx % 4) || ldx < K || ldy < N || !aligned16(x) || !aligned16(w)) return PTL_ERR_ARG;
  const int width = span_width(K), per = columns_a_split(M, N, K);
  const bool cut = per < K;
  if (cut && (parts == nullptr || !aligned16(parts))) return PTL_ERR_ARG;
  const int tiles_m = (M + F32_TILE - 1) / F32_TILE;
  const long tiles = (long)((N + F32_TILE - 1) / F32_TILE) * tiles_m;
  if (tiles > 0x3fffffff) return PTL_ERR_ARG;
  gemm_f32_tile_kernel<<<dim3((unsigned)((tiles + 7) / 8 * 8), (K + per - 1) / per), 256, 0, st>>>(
      y, x, w, M, N, K, ldx, ldy, tiles_m, (int)tiles, width, per, cut ? parts : nullptr);
  if (cut)
    gemm_f32_sum_kernel<<<(unsigned)(((long)M * N + 1023) / 1024), 256, 0, st>>>(y, parts, (K + width - 1) / width, M, N, ldy);
  return ptl_launch_status();
}
