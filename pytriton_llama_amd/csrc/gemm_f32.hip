// y = x W^T in float32 on the matrix cores: row-major x [M, K] (row stride ldx) and W [N, K],
// float32 products and sums (v_mfma_f32_*_f32 multiplies and adds in float32, so this is the same
// true 32-bit arithmetic as the vector-FMA kernel of gemm.hip, in another order).
//
// Both kernels need K % 4 == 0 and 16-byte aligned rows of x and W; everything else stays with the
// vector-FMA kernel. Inside a block of k the order of the products is free as long as both
// operands follow it, so a lane always loads four consecutive k in one 16-byte load and hands them
// to four matrix instructions one after the other.
#include "common.h"
#include "device.h"
#include "mfma_f32.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

// ===========================================================================
// Few rows of x (M <= 16, a decode step): bound by reading W once. A workgroup owns ROWS rows of W;
// its waves split K among themselves, every wave keeps up to 16 KB of W under way (two sets of U
// loads of 1 KB), and their partial sums meet in LDS. v_mfma_f32_16x16x4_f32: lane l (ln = l % 16,
// lg = l / 16) holds A[ln][k = lg] and B[k = lg][ln] and gets D[4 lg + i][ln].
//
// ROWS 16: A is 16 rows of W x 16 columns, a load instruction reads 64 bytes of each row; B the same
// columns of 16 rows of x, from L2.
// ROWS 8: with at most 8 rows of x half of such a tile would be empty, so the tile holds two blocks of
// 16 columns of the same 8 rows (lanes ln < 8 the first block, ln >= 8 the second), of W and of x
// alike. The products that matter are then D[n < 8][m < 8] and D[n >= 8][m >= 8], and every load
// instruction, of W and of x, still brings 1 KB that is used. It gives twice the workgroups. MT tiles
// of 8 rows of x share the loads of W.
//
// gemm_f32_few_kernel reads x again for every tile and takes the sums of any length;
// gemm_f32_held_kernel keeps x in registers and walks several tiles.
//
// Measured (one MI355X, cold weights, 4 rows; in brackets the vector-FMA kernel that ran first and
// gemm_f32_few_kernel): 16,384 x 2,048 25 us = 5.4 TB/s (245, 33), 2,048 x 8,192 17 us = 4.0 TB/s (928, 18.5),
// 128,256 x 2,048 171 us = 6.1 TB/s (680, 214); a decode step of 4 rows at the Llama-3.2-1B shape 1.57 ms
// (28.2, 1.78).
// ===========================================================================
template <int ROWS, int MT, int U>
__global__ void __launch_bounds__(1024)
gemm_f32_few_kernel(float* __restrict__ y, const float* __restrict__ x, const float* __restrict__ w,
                    int M, int N, int K, long ldx, long ldy, int k_per_wave) {
  extern __shared__ float red[];                 // [waves][MT][64][4]
  static_assert(ROWS == 16 || ROWS == 8, "rows of W a tile");
  constexpr int XR = ROWS;                       // rows of x in a tile
  constexpr int KB = ROWS == 8 ? 32 : 16;        // columns of W that one load instruction covers
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, ln = lane & 15, lg = lane >> 4;
  const int nwaves = blockDim.x >> 6;
  const int n0 = blockIdx.x * ROWS;
  const int koff = 4 * lg + (ROWS == 8 ? 16 * (ln >> 3) : 0);
  const float* wp = w + (size_t)min(n0 + ln % ROWS, N - 1) * K + koff;
  const float* xp[MT];
  bool xok[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = XR * t + ln % ROWS;
    xok[t] = m < M;
    xp[t] = x + (size_t)min(m, M - 1) * ldx + koff;
  }
  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int kb = wave * k_per_wave;
  const int ke = min(K, kb + k_per_wave);
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
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[u].f[s], xf[t][u].f[s], acc[t], 0, 0, 0);
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
  for (int t = 0; t < MT; ++t)
    *reinterpret_cast<f32x4*>(red + (((size_t)wave * MT + t) * 64 + lane) * 4) = acc[t];
  __syncthreads();
  // a thread a result; the sums of the waves (and of the two blocks of an 8-row tile) in order
  for (int i = threadIdx.x; i < ROWS * XR * MT; i += blockDim.x) {
    const int n = i % ROWS, m = i / ROWS, t = m / XR, j = m % XR;
    if (m >= M || n0 + n >= N) continue;
    float s = 0.f;
    for (int wv = 0; wv < nwaves; ++wv) {
      const float* p = red + ((size_t)wv * MT + t) * 256;
      s += p[((n >> 2) * 16 + j) * 4 + (n & 3)];
      if (ROWS == 8) s += p[(((n + 8) >> 2) * 16 + j + 8) * 4 + (n & 3)];
    }
    y[(size_t)m * ldy + n0 + n] = s;
  }
}

// Up to 8 rows with a wave's share of the columns in registers: x [8, 32 NB] of every wave is read once, and
// the workgroup then walks 8-row tiles of W (blockIdx.x, + gridDim.x, ...), so that W is all that is read in
// the loop: read again for every tile, x comes through the same path from L2 as W does and is as many bytes
// (128,256 x 2,048, us at 1, 4 and 8 rows: 185, 214, 254; held 165, 171, 177). The next tile's first columns are on their way while a tile's sums are
// added up, in two buffers, one barrier a tile.
template <int ROWS, int NB>
__global__ void __launch_bounds__(1024)
gemm_f32_held_kernel(float* __restrict__ y, const float* __restrict__ x, const float* __restrict__ w,
                     int M, int N, int K, long ldx, long ldy, int k_per_wave, int tiles) {
  constexpr int KB = ROWS == 8 ? 32 : 16;        // columns of a block (as above)
  constexpr int U = 4, S = NB / U;               // blocks a turn, turns a tile
  static_assert(S % 2 == 0, "the two sets of registers change places an even number of times a tile");
  extern __shared__ float red[];                 // [2][waves][64][4]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, ln = lane & 15, lg = lane >> 4;
  const int nwaves = blockDim.x >> 6;
  const int koff = 4 * lg + (ROWS == 8 ? 16 * (ln >> 3) : 0);
  const int kb = wave * k_per_wave, ke = min(K, kb + k_per_wave);
  const int left = ke - kb - koff;               // this lane's columns of block b are there if KB b < left
  F4 xf[NB];
  {
    const float* xp = x + (size_t)min(ln % ROWS, M - 1) * ldx + kb + koff;
    const bool row = ln % ROWS < M;
#pragma unroll
    for (int b = 0; b < NB; ++b) xf[b].u = row && KB * b < left ? load16(xp + KB * b) : zero16();
  }
  F4 wa[U], wb[U];
  auto load_w = [&](F4 (&f)[U], int tile, int b0) __attribute__((always_inline)) {
    const float* wp = w + (size_t)min(ROWS * tile + ln % ROWS, N - 1) * K + kb + koff;
#pragma unroll
    for (int u = 0; u < U; ++u) f[u].u = KB * (b0 + u) < left ? load_once(wp + KB * (b0 + u)) : zero16();
  };
  load_w(wa, blockIdx.x, 0);
  int at = 0;
  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x, at ^= 1) {
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
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
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(cur[u].f[i], xf[U * s + u].f[i], acc, 0, 0, 0);
    }
    float* const sums = red + at * nwaves * 256;
    *reinterpret_cast<f32x4*>(sums + (wave * 64 + lane) * 4) = acc;
    __syncthreads();
    for (int i = threadIdx.x; i < ROWS * ROWS; i += blockDim.x) {   // a thread a result, the waves' sums in order
      const int n = i % ROWS, m = i / ROWS;
      if (m < M && ROWS * tile + n < N) {
        float r = 0.f;
        for (int wv = 0; wv < nwaves; ++wv) {
          const float* p = sums + wv * 256;
          r += p[((n >> 2) * 16 + m) * 4 + (n & 3)];
          if (ROWS == 8) r += p[(((n + 8) >> 2) * 16 + m + 8) * 4 + (n & 3)];
        }
        y[(size_t)m * ldy + ROWS * tile + n] = r;
      }
    }
  }
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// M <= 16, K % 4 == 0, ldx % 4 == 0, x and w 16-byte aligned.
extern "C" int ptl_gemm_f32_few(float* y, const float* x, const float* w, int M, int N, int K, long ldx, long ldy,
                                hipStream_t st) {
  if (M <= 0 || N <= 0) return PTL_OK;
  if (M > 16 || K <= 0 || K % 4 || (M > 1 && ldx % 4) || ldx < K || ldy < N || !aligned16(x) || !aligned16(w))
    return PTL_ERR_ARG;
  // up to 8 rows 8-row tiles (gemm_f32_few_kernel, us at 4 rows, 8- against 16-row tiles: 2,048 x 2,048 7.3 / 9.5, 16,384 x 2,048
  // 31.7 / 33.0, 2,048 x 8,192 18.0 / 32.7, 128,256 x 2,048 208 / 228); beyond, where they cost a second load of
  // x, only while 16-row tiles leave a third of the compute units empty (us at 16 rows: 2,048 x 8,192 29 / 37,
  // 3,072 x 2,048 16.2 / 11.9, 16,384 x 2,048 54.6 / 39.9). At 16 rows the kernel for many rows takes 32, 18
  // and 46 us; at 32 rows this one is slower at every size.
  const int cus = compute_units();
  const int rows = M <= 8 || (N + 15) / 16 * 3 < 2L * cus ? 8 : 16;
  const long blocks = (N + rows - 1) / rows;
  // waves a workgroup: at least 256 columns each (128 in 16-row tiles), until the chip has 32 a compute unit
  // in 16-row tiles; 8-row tiles read less a wave and take four times as many
  int waves = 1;
  const int least = rows == 8 ? 256 : 128;
  while (waves < 16 && K / (waves * 2) >= least && (waves < 4 || blocks * waves < (rows == 8 ? 64L : 32L) * cus)) waves <<= 1;
  const int per = ((K + waves - 1) / waves + 31) / 32 * 32;
#define GO(ROWS, MT)                                                                                            \
  gemm_f32_few_kernel<ROWS, MT, 8 / MT><<<(unsigned)blocks, waves * 64, (size_t)waves * MT * 1024, st>>>(          \
      y, x, w, M, N, K, ldx, ldy, per)
  // x in registers where it fits, up to 512 columns a wave of 8 rows or 256 of 16, 16 waves a compute unit. In
  // 16-row tiles (us at 16 rows, read again against held): 16,384 x 2,048 43 / 35, 3,072 x 2,048 12.0 / 11.7,
  // 128,256 x 2,048 317 / 239; not where 8-row tiles are taken for more than 8 rows (2,048 x 2,048 10.0 / 11.3).
  const int most = rows == 8 ? 512 : 256;
  if (K <= 16 * most && (M <= 8 || rows == 16)) {
    const int tiles = (int)blocks;
    const int hw = max(rows == 8 ? waves : 1, (K + most - 1) / most);
    const int share = ((K + hw - 1) / hw + 31) / 32 * 32;
    const long resident = (long)cus * (16 / hw);
    const long each = (tiles + resident - 1) / resident;
    const unsigned grid = (unsigned)((tiles + each - 1) / each);
#define HELD(ROWS, NB) \
  gemm_f32_held_kernel<ROWS, NB><<<grid, hw * 64, (size_t)hw * 2048, st>>>(y, x, w, M, N, K, ldx, ldy, share, tiles)
    if (rows == 16) HELD(16, 16);
    else if (share <= 256) HELD(8, 8);
    else HELD(8, 16);
#undef HELD
    return ptl_launch_status();
  }
  if (rows == 16) GO(16, 1);
  else if (M <= 8) GO(8, 1);
  else GO(8, 2);
#undef GO
  return ptl_launch_status();
}

// ===========================================================================
// Many rows of x (a prompt portion): tiles of BN rows of W x BM rows of x a workgroup of four waves
// (two along each side), F32_BK columns of K at a time through LDS, two buffers: the next tile is on its
// way from memory to registers while this one is multiplied, one barrier a tile.
// A wave of the largest tile multiplies 64 x 64: for 8 columns it reads four 16-byte fragments a lane and
// issues 16 matrix instructions of 64 clocks each (mfma_f32.h), so the matrix cores bound it.
//
// A grid of few tiles is cut along K as well (blockIdx.y): the parts of the sums go to a workspace
// [splits, M, N] and a second kernel adds them in order.
//
// Measured (one MI355X, us; the vector-FMA kernel that ran before in brackets): 700 x 16,384 x 2,048 420 =
// 112 TFLOP/s (1,386), 700 x 2,048 x 8,192 230 (1,251), 700 x 3,072 x 2,048 100 (370), 483 x 1,536 x 2,048
// 38 (224), 64 x 2,048 x 8,192 33 (967). Relative error against 64 bits at K = 2,048: 3.7e-7 (8.1e-7).
// ===========================================================================
template <int BN, int BM>
__global__ void __launch_bounds__(256)
gemm_f32_tile_kernel(float* __restrict__ y, const float* __restrict__ x, const float* __restrict__ w,
                     int M, int N, int K, long ldx, long ldy, int tiles_m, int tiles, int k_per_split, long split_stride) {
  constexpr int TN = BN / 64, TM = BM / 64;      // 32 x 32 results of a wave along each side
  __shared__ uint4 ws[2][BN * 8];
  __shared__ uint4 xs[2][BM * 8];
  // Workgroups go to the eight XCDs in turn: each gets a run of tiles, neighbours in the run share
  // rows of W, so that W comes into one L2 once.
  const int per_xcd = (tiles + 7) / 8;
  const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (tile >= tiles || (int)(blockIdx.x >> 3) >= per_xcd) return;
  const int n0 = tile / tiles_m * BN, m0 = tile % tiles_m * BM;
  const int kb = blockIdx.y * k_per_split, ke = min(K, kb + k_per_split);
  y += (size_t)blockIdx.y * split_stride;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, lr = lane & 31, lh = lane >> 5;
  const int wn = (wave & 1) * (BN / 2), wm = (wave >> 1) * (BM / 2);
  const int piece = tid & 7, row = tid >> 3;     // of the tile's 16-byte pieces, those of rows row + 32 i
  const float* wp[BN / 32];
  const float* xp[BM / 32];
#pragma unroll
  for (int i = 0; i < BN / 32; ++i) wp[i] = w + (size_t)min(n0 + row + 32 * i, N - 1) * K + 4 * piece;
#pragma unroll
  for (int i = 0; i < BM / 32; ++i) xp[i] = x + (size_t)min(m0 + row + 32 * i, M - 1) * ldx + 4 * piece;
  uint4 wr[BN / 32], xr[BM / 32];
  auto fetch = [&](int k) {
    const bool ok = k + 4 * piece < ke;
#pragma unroll
    for (int i = 0; i < BN / 32; ++i) wr[i] = ok ? load16(wp[i] + k) : zero16();
#pragma unroll
    for (int i = 0; i < BM / 32; ++i) xr[i] = ok ? load16(xp[i] + k) : zero16();
  };
  auto put = [&](int b) {
#pragma unroll
    for (int i = 0; i < BN / 32; ++i) ws[b][f32_piece(row + 32 * i, piece)] = wr[i];
#pragma unroll
    for (int i = 0; i < BM / 32; ++i) xs[b][f32_piece(row + 32 * i, piece)] = xr[i];
  };
  f32x16_t acc[TN][TM];
#pragma unroll
  for (int a = 0; a < TN; ++a)
#pragma unroll
    for (int b = 0; b < TM; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;
  int nrow[TN], mrow[TM];
#pragma unroll
  for (int a = 0; a < TN; ++a) nrow[a] = wn + 32 * a;
#pragma unroll
  for (int c = 0; c < TM; ++c) mrow[c] = wm + 32 * c;
  fetch(kb);
  put(0);
  __syncthreads();
  int buf = 0;
  for (int k = kb; k < ke; k += F32_BK, buf ^= 1) {
    const bool more = k + F32_BK < ke;
    if (more) fetch(k + F32_BK);
    f32_multiply<TN, TM>(acc, ws[buf], xs[buf], nrow, mrow, lane);
    if (more) put(buf ^ 1);
    __syncthreads();
  }
  const bool four = (N & 3) == 0 && (ldy & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
#pragma unroll
  for (int c = 0; c < TM; ++c) {
    const int m = m0 + wm + 32 * c + lr;
    if (m >= M) continue;
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = n0 + wn + 32 * a + 8 * q + 4 * lh;
        float* at = y + (size_t)m * ldy + n;
        if (four) {
          if (n < N)
            *reinterpret_cast<float4*>(at) = make_float4(acc[a][c][4 * q], acc[a][c][4 * q + 1], acc[a][c][4 * q + 2],
                                                         acc[a][c][4 * q + 3]);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (n + i < N) at[i] = acc[a][c][4 * q + i];
        }
      }
  }
}

__global__ void __launch_bounds__(256)
gemm_f32_sum_kernel(float* __restrict__ y, const float* __restrict__ parts, int splits, int M, int N, long ldy) {
  const long total = (long)M * N;
  if ((N & 3) == 0 && (ldy & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0) {
    const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= total) return;
    float4 s = *reinterpret_cast<const float4*>(parts + i);
    for (int p = 1; p < splits; ++p) {
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
    for (int p = 0; p < splits; ++p) s += parts[(size_t)p * total + i];
    y[i / N * ldy + i % N] = s;
  }
}

// Sums of fewer products than this are added up in one order whatever the number of rows (every tile
// walks K alike), so that a request's results do not depend on what else is in its step; ops.gemm_nt
// keeps them off the kernel for few rows as well.
#define F32_ONE_ORDER_K 512

struct TilePlan {
  int bn, bm, splits;
};

// The tile and the number of cuts along K that a count of the work says are done first. The four
// waves of a workgroup take the four SIMDs of a compute unit, so what counts is the fullest unit: r
// workgroups, one after the other, at 0.5 TFLOP/s (128 TFLOP/s on 256 units), each with about two
// steps of F32_BK lost at its start and end; less than three at a time on a unit leave gaps (one alone
// takes 1.6 times as long). A cut costs the second kernel and the traffic of the partial sums.
// Against a sweep of the three tiles with 1 to 16 cuts (M 64 to 700, N 16 to 16,384, K 2,048 and
// 8,192; one MI355X) the plan is within 6 % of the fastest; without cuts 483 x 1,536 x 2,048 takes 53
// instead of 38 us, 64 x 2,048 x 8,192 takes 140 instead of 33. Sums of fewer than F32_ONE_ORDER_K products
// are never cut.
static TilePlan tile_plan(int M, int N, int K) {
  const int cus = compute_units();
  static const struct { int bn, bm; } shapes[] = {{64, 64}, {128, 64}, {128, 128}};
  TilePlan best{64, 64, 1};
  double least = 1e30;
  for (const auto& s : shapes) {
    const long tiles = (long)((N + s.bn - 1) / s.bn) * ((M + s.bm - 1) / s.bm);
    for (int splits = 1; splits <= 16; ++splits) {
      const int per = ((K + splits - 1) / splits + F32_BK - 1) / F32_BK * F32_BK;
      if (splits > 1 && (K < F32_ONE_ORDER_K || per < 4 * F32_BK || (long)per * (splits - 1) >= K)) continue;
      const double one = 2.0 * s.bn * s.bm * (per + 2 * F32_BK) / 0.5e12;
      const double r = (double)((tiles * splits + cus - 1) / cus);
      double t = one * (r < 4 ? 0.8 * (r + 1) : r + 0.3);
      if (splits > 1) t += 4e-6 + 4.0 * M * N * (splits + 1) / 6e12;
      if (t < least) {
        least = t;
        best = TilePlan{s.bn, s.bm, splits};
      }
    }
  }
  return best;
}

// floats of workspace ptl_gemm_f32 wants for these sizes (0: none)
extern "C" long ptl_gemm_f32_workspace(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const TilePlan p = tile_plan(M, N, K);
  return p.splits > 1 ? (long)p.splits * M * N : 0;
}

// K % 4 == 0, ldx % 4 == 0, x and w 16-byte aligned. ``parts``: workspace of ptl_gemm_f32_workspace(M, N, K)
// floats, 16-byte aligned (null where that is 0).
extern "C" int ptl_gemm_f32(float* y, const float* x, const float* w, int M, int N, int K, long ldx, long ldy,
                            float* parts, hipStream_t st) {
  if (M <= 0 || N <= 0) return PTL_OK;
  if (K <= 0 || K % 4 || (M > 1 && ldx % 4) || ldx < K || ldy < N || !aligned16(x) || !aligned16(w)) return PTL_ERR_ARG;
  const TilePlan p = tile_plan(M, N, K);
  if (p.splits > 1 && (parts == nullptr || !aligned16(parts))) return PTL_ERR_ARG;
  const int tiles_m = (M + p.bm - 1) / p.bm;
  const long tiles = (long)((N + p.bn - 1) / p.bn) * tiles_m;
  if (tiles > 0x3fffffff) return PTL_ERR_ARG;
  const int per = ((K + p.splits - 1) / p.splits + F32_BK - 1) / F32_BK * F32_BK;
  float* out = p.splits > 1 ? parts : y;
  const long ld = p.splits > 1 ? N : ldy;
  const dim3 grid((unsigned)((tiles + 7) / 8 * 8), p.splits);
#define GO(BN, BM)                                                                                         \
  gemm_f32_tile_kernel<BN, BM><<<grid, 256, 0, st>>>(out, x, w, M, N, K, ldx, ld, tiles_m, (int)tiles, per, \
                                                     p.splits > 1 ? (long)M * N : 0)
  if (p.bm == 128) GO(128, 128);
  else if (p.bn == 128) GO(128, 64);
  else GO(64, 64);
#undef GO
  if (p.splits > 1)
    gemm_f32_sum_kernel<<<(unsigned)(((long)M * N + 1023) / 1024), 256, 0, st>>>(y, parts, p.splits, M, N, ldy);
  return ptl_launch_status();
}
