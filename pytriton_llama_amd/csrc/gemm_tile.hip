// Products of some hundred rows of x (a batch of short prompts, a portion of a prompt beside decoding requests) in
// bfloat16 on the matrix cores, where the library's product is far from what the card can do: x [M, K] times the
// row-major W [N, K], transposed.
//   ptl_tile_gemm_sums   the product as float32 partial sums over equal slices of K, which the norm that follows
//                        adds up (ptl_rows_sum_add_rmsnorm): a matrix of few rows and a deep K (the down and output
//                        projections) has too few tiles for the compute units otherwise
//   ptl_tile_gate_up     act(x Wg^T) * (x Wu^T) for W = [Wg; Wu]: the rows of a gate and of its up lie in one wave's
//                        tile, so the [M, 2 I] product is never stored
//   ptl_tile_qkv_rope_store  q | k | v: the two rows of W of a rotated pair lie in one wave's tile; q is stored rotated, k (rotated)
//                        and v go to their pages
// The reference runs these products through cuBLAS and the rest as kernels of their own
// (lite_llama/models/llama.py:107-120, lite_llama/kernels/swiglu.py, skip_rmsnorm.py).
//
// Four waves multiply, each a part of the tile, and four bring the operands through LDS (tile_stream.h). What bounds it: with
// few workgroups the latency of W on its way from HBM (a chunk a compute unit and 0.35 to 0.7 us, of which the matrix
// instructions take 0.06 to 0.5), with all compute units at work what they read from L2, 11 to 16 TB/s. LDS is next: a
// wave of 64 x 64 reads as many bytes as LDS gives in the time of its products, hence parts of 64 x 128 and 144 x 64 in the
// larger tiles. The reads go between the products (tile_interleave), a workgroup walks several tiles where there are more than the chip
// holds, and the loading waves run ahead into the next one.
// Tried: W from the blocked copy straight into registers, x alone through LDS (2,048 x 2,048 x 8,192: 150 us for
// 128 x 256, 85 for 128 x 128, against 103 and 67); a seventh wave that touches W 6 to 16 chunks ahead (10 to 35 % slower);
// rows of x and W padded by 64 or 128 columns (level).
//
// Measured (one MI355X, cold weights, us, a product over and over in a recorded graph, which flatters the library against a step, where it shares
// the caches with others: ops/kernels.py has the times in a step; the library's product and the kernel behind it in brackets): down projection with
// sum, residual and norm, 2,048 x 8,192, 80 / 285 / 532 / 1,024 rows: 17.6 / 27.0 / 32.6 / 50.6 (24.6 / 36.2 / 47.8 / 55.2);
// 3,072 x 8,192 20.8 / 34.8 / 44.2 / 63.2 (43.8 / 38.5 / 54.8 / 72.5); 4,096 x 14,336 32.1 / 52.7 / 74.2 / 120 (47.4 / 83.2 /
// 120 / 139); output projection, 2,048 x 2,048 10.0 / 16.1 / 18.5 / 21.1 (11.5 / 14.1 / 17.1 / 21.3). Gate-up with SiLU-multiply,
// 2 x 8,192 x 2,048, 80 / 285 / 532 / 700 rows: 20.5 / 29.6 / 40.7 / 54.3 (22.4 / 34.2 / 47.3 / 53.5). q | k | v with rotation and cache
// write, 3,072 x 2,048 at 277 / 532 / 1,024 / 2,048 rows 11.8 / 15.9 / 25.3 / 31.8 (18.5 / 22.4 / 30.2 / 37.1), 5,120 x 3,072 at 277 /
// 532 / 1,024 20.9 / 29.8 / 45.1 (26.5 / 33.0 / 46.7), 6,144 x 4,096 28.9 / 39.0 / 53.6 (35.1 / 46.4 / 61.6).
// What bounds the loads: a compute unit has some 64 KB under way, which come back in order, so what lies in L2 waits for what comes from
// HBM: 160 rows of x and 128 of W a tile, 277 x 16,384 x 2,048, loads alone 24 us (the whole product 28.6), 14 with W in the
// memory-side cache, whatever the depth, the layout of W or the kind of load; x alone 26 TB/s from L2. Products alone 18 us.
// W fetched ahead through the scalar cache: 24 -> 31 us.
#include "common.h"
#include "device.h"
#include "mfma.h"
#include "tile_stream.h"

namespace {

enum { OUT_SUMS = 0, OUT_GLU = 1, OUT_QKV = 2 };

constexpr int KC = TILE_ROW / 2;           // columns of a chunk

// round to nearest even by the hardware's conversion
__device__ __forceinline__ bf16_t to_bf16(float f) {
  union { __bf16 b; bf16_t u; } r;
  r.b = (__bf16)f;
  return r.u;
}
__device__ __forceinline__ float rounded(float f) { return (float)(__bf16)f; }

// The activation of a pair, as the other kernels for a gate and its up row have it (glu); TILE_SILU_HW: SiLU by the
// hardware's exponential and reciprocal, a few units in the last place of float32 in front of the rounding to bfloat16,
// as silu_mul has it (activation.hip). The matrix cores stand still meanwhile: 2,048 x 16,384 x 2,048 takes 136 us so and
// 150 with expf and a division. It is the caller who says that it had the one or the other before.
constexpr int TILE_SILU_HW = 16;
__device__ __forceinline__ float pair_value(const GluArgs& a, float g, float u) {
  if (a.act == TILE_SILU_HW)
    return g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * g)) * u;
  return glu(a, g, u);
}

// Where q | k | v go (ptl_tile_qkv_rope_store).
struct QkvArgs {
  const float2* const* turns;      // where it says where the cosines and sines [M][D / 2] lie, or null
  const int32_t* slots;
  bf16_t *k_cache, *v_cache;
  int Hq, Hkv, D, page_size;
  long ldq;
};

struct TileArgs {
  void* y;                   // OUT_SUMS: float32 [splits, M, N]; OUT_GLU: bfloat16 [M, N]; OUT_QKV: q
  const bf16_t* x;
  const bf16_t* w;
  int M, N, K;               // N: columns of y (OUT_QKV: pairs of columns of q | k | v)
  long ldx;
  int splits, tiles_m, tiles_n;
  GluArgs act;
  QkvArgs qkv;
};

struct Tile {
  int m0, n0, split;
};

// Tile t of the list: slices of K slowest; then groups of eight tiles of rows, inside which the rows go fastest, so
// that consecutive tiles share rows of W and of x.
template <int BM, int COLS> __device__ __forceinline__ Tile tile_at(const TileArgs& a, int t) {
  constexpr int GM = 8;
  const int per_split = a.tiles_m * a.tiles_n;
  Tile r;
  r.split = t / per_split;
  const int u = t - r.split * per_split;
  const int group = u / (GM * a.tiles_n), in_group = u - group * (GM * a.tiles_n);
  const int gm = min(GM, a.tiles_m - group * GM);
  const int tn = in_group / gm;
  r.m0 = (group * GM + in_group - tn * gm) * BM;
  r.n0 = tn * COLS;
  return r;
}

// BM x BN: rows of x and of W a tile; WGM x WGN waves share it; NB buffers, PW loading waves.
template <int BM, int BN, int WGM, int WGN, int NB, int PW, int MODE>
__global__ void __launch_bounds__(64 * (WGM * WGN + PW))
gemm_tile_kernel(const TileArgs a) {
  constexpr int WAVES = WGM * WGN;
  constexpr int WM = BM / WGM, WN = BN / WGN;                // the wave's part of the tile
  constexpr int TM = WM / 16, TN = WN / 16;
  constexpr bool PAIRS = MODE != OUT_SUMS;                   // rows of W that meet in a result: half a wave's each
  constexpr int COLS = PAIRS ? BN / 2 : BN;                  // columns of y a tile gives
  constexpr int CHUNK = (BM + BN) * TILE_ROW;                // rows of x, then rows of W
  static_assert(!PAIRS || TN % 2 == 0, "the two of a pair meet in a wave");
  extern __shared__ __align__(16) unsigned char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int M = a.M, N = a.N, K = a.K;
  // Workgroups go to the XCDs in turn; XCD c takes a run of consecutive tiles of every round, which share rows of x
  // and of W in its L2.
  const int total = a.tiles_m * a.tiles_n * a.splits, G = gridDim.x;
  const int run = G >> 3, rest = G & 7, xcd = blockIdx.x & 7;
  const int first_tile = xcd * run + min(xcd, rest) + (blockIdx.x >> 3);
  const int my_tiles = (total - first_tile + G - 1) / G;     // (the grid has no more workgroups than there are tiles)
  const int k_per_split = K / a.splits, chunks = k_per_split / KC;
  const float2* const table = MODE == OUT_QKV && a.qkv.turns ? *a.qkv.turns : nullptr;

  if (wave >= WAVES) {
    tile_bring<BM + BN, NB, PW>(lds, wave - WAVES, lane, my_tiles, chunks, [&](int i, int r) {
      const Tile t = tile_at<BM, COLS>(a, first_tile + i * G);
      const size_t k0 = (size_t)t.split * k_per_split;
      if (r < BM) return reinterpret_cast<const char*>(a.x + (size_t)min(t.m0 + r, M - 1) * a.ldx + k0);
      const int q = r - BM;
      int row;
      if (PAIRS) {                                           // a wave's rows: one half gate, the other half up
        const int part = q / WN, at = q - part * WN, up = at >= WN / 2;
        row = min(t.n0 + part * (WN / 2) + (up ? at - WN / 2 : at), N - 1);
        if (MODE == OUT_QKV) {                               // ... one half of a head and the other
          const int half = a.qkv.D >> 1, head = row / half;
          row += head * half + (up ? half : 0);
        } else {
          row += up ? N : 0;
        }
      } else {
        row = min(t.n0 + q, N - 1);
      }
      return reinterpret_cast<const char*>(a.w + (size_t)row * K + k0);
    });
    return;
  }

  const int ln = lane & 15, lg = lane >> 4, wm = wave / WGN, wn = wave - wm * WGN;
  const int x_at = (wm * WM + ln) * TILE_ROW, w_at = (BM + wn * WN + ln) * TILE_ROW;
  const int p0 = 16 * (lg ^ (ln & 7)), p1 = 16 * ((4 + lg) ^ (ln & 7));
  f32x4_t acc[TN][TM];
  Frag8 xf[2][TM], wf[2][TN];                                // of the two halves of a chunk
  auto read = [&](const unsigned char* at, int h) __attribute__((always_inline)) {
    const int p = h ? p1 : p0;
#pragma unroll
    for (int j = 0; j < TN; ++j) wf[h][j].u = load16(at + w_at + j * 16 * TILE_ROW + p);
#pragma unroll
    for (int i = 0; i < TM; ++i) xf[h][i].u = load16(at + x_at + i * 16 * TILE_ROW + p);
  };
  auto multiply = [&](int h) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h][j].v, xf[h][i].v, acc[j][i], 0, 0, 0);
  };
  int slot = 0;
  for (int n = 0; n < my_tiles; ++n) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    tile_meet();
    read(lds + slot * CHUNK, 0);
    for (int c = 0; c + 1 < chunks; ++c) {
      tile_wait_lds();
      __builtin_amdgcn_sched_barrier(0);
      read(lds + slot * CHUNK, 1);
      multiply(0);
      tile_interleave<TM + TN, TM * TN>();
      tile_wait_lds();             // every read of the chunk has come back before the wave says that it is done with it
      tile_meet();
      slot = slot + 1 == NB ? 0 : slot + 1;
      __builtin_amdgcn_sched_barrier(0);
      read(lds + slot * CHUNK, 0);
      multiply(1);
      tile_interleave<TM + TN, TM * TN>();
    }
    tile_wait_lds();
    __builtin_amdgcn_sched_barrier(0);
    read(lds + slot * CHUNK, 1);
    multiply(0);
    tile_interleave<TM + TN, TM * TN>();
    tile_wait_lds();
    multiply(1);
    slot = slot + 1 == NB ? 0 : slot + 1;

    // the lane holds, of every 16 x 16 results, the columns 4 lg + i (rows of W) of row ln (of x)
    const Tile t = tile_at<BM, COLS>(a, first_tile + n * G);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = t.m0 + wm * WM + 16 * i + ln;
      if (m >= M) continue;
      if (MODE == OUT_SUMS) {
        float* row = reinterpret_cast<float*>(a.y) + ((size_t)t.split * M + m) * N;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int col = t.n0 + wn * WN + 16 * j + 4 * lg;
          if (col < N) *reinterpret_cast<f32x4_t*>(row + col) = acc[j][i];
        }
      } else if (MODE == OUT_QKV) {
        const int half = a.qkv.D >> 1, slot = a.qkv.slots ? a.qkv.slots[m] : -1;
        const int page = slot / a.qkv.page_size, off = slot - page * a.qkv.page_size;
#pragma unroll
        for (int j = 0; j < TN / 2; ++j) {
          const int pair = t.n0 + wn * (WN / 2) + 16 * j + 4 * lg, head = pair / half, at = pair - head * half;
          if (pair >= N) continue;
          const int kv = head - a.qkv.Hq, v = kv >= a.qkv.Hkv;
          if (kv >= 0 && slot < 0) continue;
          const bool turned = !v && table;
          f32x4_t c01 = f32x4_t{1.f, 0.f, 1.f, 0.f}, c23 = c01;    // cosine, sine of two pairs
          if (turned) {
            const f32x4_t* cs = reinterpret_cast<const f32x4_t*>(table + (size_t)m * half + at);
            c01 = cs[0];
            c23 = cs[1];
          }
          union { uint2 u; bf16_t e[4]; } lo, hi;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const float c = k < 2 ? c01[2 * k] : c23[2 * k - 4], s = k < 2 ? c01[2 * k + 1] : c23[2 * k - 3];
            const float x1 = rounded(acc[j][i][k]), x2 = rounded(acc[j + TN / 2][i][k]);
            // (a copy where nothing is turned: times 1 less times 0 is a NaN beside an infinity)
            lo.e[k] = to_bf16(turned ? x1 * c - x2 * s : x1);
            hi.e[k] = to_bf16(turned ? x2 * c + x1 * s : x2);
          }
          bf16_t* to = kv < 0 ? reinterpret_cast<bf16_t*>(a.y) + (size_t)m * a.qkv.ldq + (size_t)head * a.qkv.D
                              : (v ? a.qkv.v_cache : a.qkv.k_cache) +
                                    (((size_t)page * a.qkv.Hkv + (v ? kv - a.qkv.Hkv : kv)) * a.qkv.page_size + off) * a.qkv.D;
          *reinterpret_cast<uint2*>(to + at) = lo.u;
          *reinterpret_cast<uint2*>(to + at + half) = hi.u;
        }
      } else {
        bf16_t* row = reinterpret_cast<bf16_t*>(a.y) + (size_t)m * N;
#pragma unroll
        for (int j = 0; j < TN / 2; ++j) {
          const int col = t.n0 + wn * (WN / 2) + 16 * j + 4 * lg;
          if (col >= N) continue;
          union { uint2 u; bf16_t e[4]; } o;
          // the two products are rounded to bfloat16 first, as a stored product is
#pragma unroll
          for (int k = 0; k < 4; ++k)
            o.e[k] = to_bf16(pair_value(a.act, rounded(acc[j][i][k]), rounded(acc[j + TN / 2][i][k])));
          *reinterpret_cast<uint2*>(row + col) = o.u;
        }
      }
    }
  }
}

// The tiles there are: rows of x and of W, waves along either, buffers, workgroups a compute unit (LDS), and what one
// takes, in us: r rounds of workgroups with c chunks each, of which a share f of the chip's places is taken, take
// r (c (chunk + full f) + tile). Fitted to 12 shapes of W (2,048 to 28,672 rows, 2,048 to 14,336 columns), 80 to 2,048 rows and
// 1 to 8 slices with two loading waves. Against the times with four (11 shapes, 80 to 1,024 rows, recorded): 15 to 22 % off
// (root mean square, each tile's by much the same, which does not change the choice); the plan chosen by it is 1.7 % slower on
// average than the fastest, 8.5 % at worst.
#define TILES(T)                                     \
  T(64, 64, 2, 2, 5, 2, 0.17f, 0.30f, 1.4f)          \
  T(64, 128, 2, 2, 5, 1, 0.30f, 0.08f, 1.9f)         \
  T(128, 64, 2, 2, 5, 1, 0.27f, 0.09f, 2.1f)         \
  T(96, 128, 2, 2, 5, 1, 0.35f, 0.10f, 2.7f)         \
  T(128, 128, 2, 2, 4, 1, 0.35f, 0.19f, 4.1f)        \
  T(160, 128, 2, 2, 4, 1, 0.40f, 0.20f, 4.8f)        \
  T(192, 128, 2, 2, 3, 1, 0.43f, 0.29f, 5.8f)        \
  T(128, 192, 2, 2, 3, 1, 0.47f, 0.27f, 5.5f)        \
  T(96, 256, 2, 2, 3, 1, 0.56f, 0.23f, 5.2f)         \
  T(112, 256, 1, 4, 3, 1, 0.59f, 0.26f, 6.1f)        \
  T(128, 256, 2, 2, 3, 1, 0.59f, 0.35f, 7.3f)        \
  T(144, 256, 1, 4, 3, 1, 0.67f, 0.27f, 7.6f)

constexpr int LOADERS = 4;                       // loading waves (with two of them 1 to 4 % slower: tile_stream.h)

struct Shape {
  int rows, cols, per_unit;
  float chunk, full, tile;
};
constexpr Shape SHAPES[] = {
#define T(BM, BN, WGM, WGN, NB, OCC, CHUNK, FULL, TILE) {BM, BN, OCC, CHUNK, FULL, TILE},
    TILES(T)
#undef T
};
constexpr int N_SHAPES = sizeof(SHAPES) / sizeof(SHAPES[0]);

struct Plan {
  int shape, splits;
  float us;
};

// rows_w: rows of W. Slices are equal, of at least 512 columns, at most eight; each costs the float32 sums once more on their
// way out and in (5 TB/s).
Plan plan_for(int M, int rows_w, int K, bool sums) {
  const int cus = compute_units();
  Plan best{0, 1, 1e30f};
  for (int s = 1; s <= (sums ? 8 : 1); s *= 2) {
    if ((K / KC) % s || (s > 1 && K / s < 512)) break;
    const float extra = s > 1 ? 4.0f * s * M * rows_w / 5e6f : 0.f;
    for (int i = 0; i < N_SHAPES; ++i) {
      const Shape& h = SHAPES[i];
      const long tiles = (long)((M + h.rows - 1) / h.rows) * ((rows_w + h.cols - 1) / h.cols) * s;
      const long places = (long)h.per_unit * cus, rounds = (tiles + places - 1) / places;
      const float fill = (float)tiles / (float)(rounds * places);
      const float us = rounds * (K / KC / s * (h.chunk + h.full * fill) + h.tile) + extra;
      if (us < best.us) best = Plan{i, s, us};
    }
  }
  return best;
}

template <int BM, int BN, int WGM, int WGN, int NB, int OCC, int MODE>
int launch(TileArgs a, hipStream_t stream) {
  const size_t lds = (size_t)NB * (BM + BN) * TILE_ROW;
  auto kernel = gemm_tile_kernel<BM, BN, WGM, WGN, NB, LOADERS, MODE>;
  static LdsAllowance allowance;
  if (!allowance.ask(reinterpret_cast<const void*>(kernel), lds)) return PTL_ERR_LAUNCH;
  const int cols = MODE == OUT_SUMS ? BN : BN / 2;
  a.tiles_m = (a.M + BM - 1) / BM;
  a.tiles_n = (a.N + cols - 1) / cols;
  const long total = (long)a.tiles_m * a.tiles_n * a.splits, most = (long)OCC * compute_units();
  if (total > 0x3fffffff) return PTL_ERR_ARG;
  kernel<<<(unsigned)(total < most ? total : most), 64 * (WGM * WGN + LOADERS), lds, stream>>>(a);
  return ptl_launch_status();
}

template <int MODE> int run(int shape, const TileArgs& a, hipStream_t stream) {
  int i = 0;
#define T(BM, BN, WGM, WGN, NB, OCC, CHUNK, FULL, TILE) \
  if (shape == i++) return launch<BM, BN, WGM, WGN, NB, OCC, MODE>(a, stream);
  TILES(T)
#undef T
  return PTL_ERR_ARG;
}

bool aligned(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

bool bad(const void* y, const void* x, const void* w, int M, int N, int K, long ldx) {
  return M <= 0 || N <= 0 || N % 4 || K <= 0 || K % KC || ldx % 8 || ldx < K || !aligned(y) || !aligned(x) || !aligned(w);
}

}  // namespace

extern "C" int ptl_tile_shapes() { return N_SHAPES; }

// The slices of K that ptl_tile_gemm_sums should leave partial sums of.
extern "C" int ptl_tile_gemm_splits(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0 || K % KC) return 1;
  return plan_for(M, N, K, true).splits;
}

// The products in a tile of the caller's (an index below ptl_tile_shapes()), for tests; the two entries behind it take the
// plan's. sums != 0: as ptl_tile_gemm_sums, in ``splits`` slices of whole chunks; else as ptl_tile_gate_up (N: I).
extern "C" int ptl_tile_product(void* y, const void* x, const void* w, int M, int N, int K, long ldx, int sums, int tile,
                                int splits, int act, float limit, hipStream_t stream) {
  if (bad(y, x, w, M, N, K, ldx) || splits < 1 || (K / KC) % splits) return PTL_ERR_ARG;
  TileArgs a{y, (const bf16_t*)x, (const bf16_t*)w, M, N, K, ldx, splits, 0, 0, GluArgs{act, limit}, QkvArgs{}};
  if (sums) return run<OUT_SUMS>(tile, a, stream);
  if (splits != 1 || !(glu_ok(act) || act == TILE_SILU_HW)) return PTL_ERR_ARG;
  return run<OUT_GLU>(tile, a, stream);
}

// y float32 [splits, M, N] = x [M, K] W^T, one slice of K each (``splits`` as ptl_tile_gemm_splits says).
// K a multiple of 64, N of 4, 16-byte aligned rows.
extern "C" int ptl_tile_gemm_sums(float* y, const void* x, const void* w, int M, int N, int K, long ldx, int splits,
                                  hipStream_t stream) {
  if (bad(y, x, w, M, N, K, ldx)) return PTL_ERR_ARG;
  const Plan p = plan_for(M, N, K, true);
  if (splits != p.splits) return PTL_ERR_ARG;
  return ptl_tile_product(y, x, w, M, N, K, ldx, 1, p.shape, p.splits, GLU_SILU, 0.f, stream);
}

// out bfloat16 [M, I] = act(x Wg^T) * (x Wu^T) for W = [Wg; Wu] [2 I, K]. K a multiple of 64, I of 4, 16-byte aligned rows.
// hw_silu != 0: act is SiLU, by the hardware's functions (pair_value).
extern "C" int ptl_tile_gate_up(void* out, const void* x, const void* w, int M, int I, int K, long ldx, int act,
                                float limit, int hw_silu, hipStream_t stream) {
  if (bad(out, x, w, M, I, K, ldx) || !glu_ok(act) || (hw_silu && act != GLU_SILU)) return PTL_ERR_ARG;
  return ptl_tile_product(out, x, w, M, I, K, ldx, 0, plan_for(M, 2 * I, K, false).shape, 1, hw_silu ? TILE_SILU_HW : act,
                          limit, stream);
}

// q, k, v = x W^T (rows of W: q | k | v, heads of D), q and k rotated by a table of cosines and sines (pairs of floats [M][D / 2],
// 16-byte aligned; ``turns``: the place in device memory that holds its address, null: not at all): q [M, ldq], k and v into pages [pages, Hkv, page_size, D] at slots[m] = page * page_size + offset (below 0,
// or slots null: nowhere). The products are rounded to bfloat16 before the rotation, as stored ones are (rope.hip). K a multiple of
// 64, D of 32, 16-byte aligned rows, tables and pages. tile: -1: the plan's, else one of the caller's, for tests (two more than ptl_tile_shapes()).
extern "C" int ptl_tile_qkv_rope_store(void* q, long ldq, const void* x, const void* w, int M, int K, long ldx, const void* turns,
                                       const int32_t* slots, void* k_cache, void* v_cache, int Hq, int Hkv, int D,
                                       int page_size, int tile, hipStream_t stream) {
  if (Hq <= 0 || Hkv <= 0 || D <= 0 || D % 32 || page_size <= 0 || (long)(Hq + 2 * Hkv) * D > 0x3fffffff) return PTL_ERR_ARG;
  const int rows_w = (Hq + 2 * Hkv) * D;
  if (bad(q, x, w, M, rows_w / 2, K, ldx) || ldq % 8 || ldq < (long)Hq * D || (uintptr_t)turns % 8 || !aligned(k_cache) ||
      !aligned(v_cache) || (slots && (!k_cache || !v_cache)) || tile < -1 || tile >= N_SHAPES + 2)
    return PTL_ERR_ARG;
  const TileArgs a{q, (const bf16_t*)x, (const bf16_t*)w, M, rows_w / 2, K, ldx, 1, 0, 0, GluArgs{},
                   QkvArgs{(const float2* const*)turns, slots, (bf16_t*)k_cache, (bf16_t*)v_cache, Hq, Hkv, D, page_size, ldq}};
  // Few rows of a narrow W: the smallest tiles as long as each finds a compute unit of its own. 3,072 x 2,048 at 48 / 64 / 96 / 128
  // rows 9.6 / 9.6 / 10.3 / 10.6 us (tiles of 64 x 64 12.5 / 13.3 / 11.8 / 13.2), 5,120 x 3,072 at 48 / 64 13.8 / 14.5 (16.3 /
  // 17.4), 6,144 x 4,096 17.3 / 18.1 (20.7 / 22.1); beyond one tile a unit 5,120 x 3,072 at 80 rows 18.3 (15.0).
  const int units = compute_units(), cols = (rows_w + 31) / 32;
  if (tile == N_SHAPES || (tile < 0 && (M + 31) / 32 * cols <= units)) return launch<32, 32, 2, 1, 5, 2, OUT_QKV>(a, stream);
  if (tile == N_SHAPES + 1 || (tile < 0 && (M + 63) / 64 * cols <= units)) return launch<64, 32, 4, 1, 5, 2, OUT_QKV>(a, stream);
  return run<OUT_QKV>(tile < 0 ? plan_for(M, rows_w, K, false).shape : tile, a, stream);
}
