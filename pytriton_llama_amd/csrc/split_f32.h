// float32 products on the bfloat16 matrix cores, which do sixteen times the work of the float32 ones in the same time.
//
// A float32 number has 24 significant bits, a bfloat16 one 8, with the same exponents: x = h + m + l, h = x rounded to
// bfloat16, m = x - h rounded, l = x - h - m, and nothing is lost (h takes 8 bits, what is left of the 24 has 16 and a
// sign, m takes 8 of them, l the other 8). A product of two numbers is then nine products, each exact in float32 (8 x 8
// bits); the three smallest, m l, l m and l l, are at most 2^-23 of the whole and typically 2^-26, less than the 2^-24 that one
// addition in float32 rounds off, and are left out. (The splitting of float32 into three bfloat16 parts: Henry, Tang and
// Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations", 2019.)
// The six that are kept are added by the matrix cores from the smallest up, over a block of 32 columns; the blocks' sums
// are added to the result by vector instructions. A float32 matrix instruction rounds its sum every four columns, this one
// every 32.
//
// What is lost: the last bits of numbers below 2^-110 are too small for bfloat16, and products below 2^-126 for the matrix cores. Sums of
// 2,048 products with numbers around one, error in 2^-24 of the sum of magnitudes: 4 for numbers of about 2^-114 as for large ones, 6 for
// 2^-116, 8 to 14 for 2^-118, 30 to 80 for 2^-120; at most 2.8 times 2^-126 in all.
//
// What is not finite: inf - inf in the split makes a NaN of every sum that an infinite (or nearly infinite) number enters.
// A result that is not finite is worked out again by plain_dots.
//
// v_mfma_f32_16x16x32_bf16: lane l (ln = l % 16, lg = l / 16) holds eight columns of A[ln] and of B[ln] and gets
// D[4 lg + i][ln]. Which columns a lane group holds is free as long as A and B agree: here 4 lg .. + 3 and 16 + 4 lg .. + 3,
// which are two loads of 16 bytes that read whole 64-byte pieces of a row.
#pragma once
#include <hip/hip_runtime.h>

#include "common.h"
#include "mfma.h"
#include "mfma_f32.h"

#define SPLIT_BK 32                    // columns of a block

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

struct Split {
  Frag8 h, m, l;
};

// two numbers rounded to bfloat16, the first in the low half
__device__ __forceinline__ uint32_t two_bf16(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{a, b}), bf16x2_t));
}

__device__ __forceinline__ void split2(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = two_bf16(a, b);
  a -= __uint_as_float(h << 16);
  b -= __uint_as_float(h & 0xffff0000u);
  m = two_bf16(a, b);
  a -= __uint_as_float(m << 16);
  b -= __uint_as_float(m & 0xffff0000u);
  l = two_bf16(a, b);
}

__device__ __forceinline__ Split split8(const F4& a, const F4& b) {
  Split s;
  split2(a.f[0], a.f[1], s.h.u.x, s.m.u.x, s.l.u.x);
  split2(a.f[2], a.f[3], s.h.u.y, s.m.u.y, s.l.u.y);
  split2(b.f[0], b.f[1], s.h.u.z, s.m.u.z, s.l.u.z);
  split2(b.f[2], b.f[3], s.h.u.w, s.m.u.w, s.l.u.w);
  return s;
}

// step 0 .. 5 of a block's products: which parts of A and of B, from the smallest up
template <int STEP> __device__ __forceinline__ f32x4_t split_step(const Split& a, const Split& b, f32x4_t t) {
  const Frag8& p = STEP == 0 ? a.l : STEP == 2 || STEP == 3 ? a.m : a.h;
  const Frag8& q = STEP == 1 ? b.l : STEP == 2 || STEP == 4 ? b.m : b.h;
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(p.v, q.v, t, 0, 0, 0);
}

__device__ __forceinline__ f32x4_t split_dot(const Split& a, const Split& b) {
  f32x4_t t = {0.f, 0.f, 0.f, 0.f};
  t = split_step<0>(a, b, t);
  t = split_step<1>(a, b, t);
  t = split_step<2>(a, b, t);
  t = split_step<3>(a, b, t);
  t = split_step<4>(a, b, t);
  return split_step<5>(a, b, t);
}

__device__ __forceinline__ bool is_finite(float v) { return (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u; }

// The sums of products that the lanes with ``want`` have of their row of x and their row of W (K columns in steps of 4, 16-byte
// aligned), in float32; the other lanes keep v. The whole wave calls, and makes one sum after the other: a lane takes every
// 64th 16-byte piece of the rows (EACH of them under way, which the bits do not depend on), and the lanes' sums meet in a butterfly, so that the bits depend on the two rows alone. A
// row with a NaN in it is found with the first of its sums and gives NaN to all others that want it; nan_x keeps that of this
// lane's row of x for the caller's next call. Where such a sum is wanted is rare, and its cost has to be bounded: a NaN in
// one request's row reaches every result of that row in all products that follow. (One MI355X, us, 300 x 2,048 x 2,048 with a NaN,
// with an infinity in one row of x, and without: 46, 734, 43; 4 x 16,384 x 2,048 42, 188, 34. By the lane that
// owns the result, one column after the other: 1,133 and 705 with either. An infinity costs a sum of 2 to 3 us for every result of its row.)
template <int EACH = 2> __device__ __forceinline__ float plain_dots(float v, bool want, const float* x, const float* w, int K, bool& nan_x) {
  // (The lane and the NaN are made of a zero that the compiler does not know: worked out ahead of the loop around such a call
  // they take registers that a kernel with loads under way does not have, and their way back from memory waits for those
  // loads: gate-up of one row 28.4 -> 32.9 us.)
  unsigned zero = 0;
  asm volatile("" : "+s"(zero));
  const int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, zero));
  const float nan = __uint_as_float(0x7fc00000u + zero);
  if (want && nan_x) {
    v = nan;
    want = false;
  }
  for (unsigned long long left = __ballot(want); left; left = __ballot(want)) {
    const int owner = __builtin_ctzll(left);
    auto of_owner = [&](const float* p) __attribute__((always_inline)) {
      const uint64_t b = reinterpret_cast<uint64_t>(p);
      const uint32_t lo = __builtin_amdgcn_readlane((int)b, owner), hi = __builtin_amdgcn_readlane((int)(b >> 32), owner);
      return reinterpret_cast<const float*>((uint64_t)hi << 32 | lo);
    };
    const float *xr = of_owner(x), *wr = of_owner(w);
    float s = 0.f;
    bool nan_in_x = false, nan_in_w = false;
#pragma unroll 1
    for (int k0 = 0; k0 < K; k0 += 256 * EACH) {
      F4 a[EACH], b[EACH];
#pragma unroll
      for (int h = 0; h < EACH; ++h) {
        const int k = k0 + 256 * h + 4 * lane;
        a[h].u = k < K ? load16(xr + k) : zero16();
        b[h].u = k < K ? load16(wr + k) : zero16();
      }
#pragma unroll
      for (int h = 0; h < EACH; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          nan_in_x = nan_in_x || a[h].f[i] != a[h].f[i];
          nan_in_w = nan_in_w || b[h].f[i] != b[h].f[i];
          s = fmaf(a[h].f[i], b[h].f[i], s);
        }
      if (__any(s != s)) break;                  // (no later product makes a number of it)
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
      s += __int_as_float(__builtin_amdgcn_ds_bpermute(4 * (lane ^ o), __float_as_int(s)));
    if (lane == owner) {
      v = s;
      want = false;
    }
    if (__any(nan_in_x) && x == xr) {
      nan_x = true;
      if (want) v = nan;
      want = false;
    }
    if (__any(nan_in_w) && w == wr) {
      if (want) v = nan;
      want = false;
    }
  }
  return v;
}

// Tiles of 64 TA rows of W (or TA times 64 rows of different matrices) x 16 TC rows of x, a workgroup of four waves. A wave
// takes 16 TA rows of W, which no other wave wants, straight from memory into registers and splits them there, and all rows
// of x, which all waves want: split once, they lie in LDS as three matrices of bfloat16, two buffers of a block of 32 columns.
// Memory is three blocks ahead of the products, in registers, LDS one; one barrier a block.
//
// In LDS a row's part is four 16-byte pieces, piece lg what lane group lg multiplies; they are permuted by (row / 2) % 4, so
// that eight neighbouring lanes touch every bank once, writing along a row and reading down a column of pieces.
template <int TC> struct SplitX {
  static constexpr int ROWS = 16 * TC;
  static_assert(ROWS % 64 == 0, "every thread brings as much");
  static constexpr int EACH = ROWS / 64;                   // pieces of a block a thread brings: of rows 64 apart
  static constexpr int PIECES = 4 * ROWS;                  // of one part of a block
  static constexpr int LDS = 2 * 3 * PIECES;               // uint4
};

__device__ __forceinline__ int split_piece(int row, int lg) { return 4 * row + (lg ^ ((row >> 1) & 3)); }

// wp[a]: this lane's row of W (ln) of the wave's a-th 16, xp[i]: row threadIdx.x / 4 + 64 i of x; both at column 0. Columns
// kb .. ke, kb a multiple of the block. done(k, acc): called when the sums of a span are complete, k one past its last block's
// first column; it has to leave zeros. ``width``: columns of a span, a multiple of the block. ``groups``: of the TC 16 rows of x those that
// are wanted, the first ones (of the workgroup).
template <int TA, int TC, typename Done>
__device__ __forceinline__ void split_tile(uint4* __restrict__ lds, const float* const (&wp)[TA],
                                           const float* const (&xp)[SplitX<TC>::EACH], int kb, int ke, int width,
                                           f32x4_t (&acc)[TA][TC], Done done, int groups = TC) {
  constexpr int EACH = SplitX<TC>::EACH, PIECES = SplitX<TC>::PIECES;
  const int tid = threadIdx.x, lane = tid & 63, ln = lane & 15, lg = lane >> 4;
  const int xrow = tid >> 2, xlg = tid & 3;
  F4 wr[2][TA][2], xr[2][EACH][2];
  // (no branches here: behind one the compiler does not know how many loads are under way, and waits for all)
  auto fetch = [&](int r, int k) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int kw = min(k + 16 * h + 4 * lg, ke - 4), kx = min(k + 16 * h + 4 * xlg, ke - 4);
#pragma unroll
      for (int a = 0; a < TA; ++a) wr[r][a][h].u = load16(wp[a] + kw);
#pragma unroll
      for (int i = 0; i < EACH; ++i) xr[r][i][h].u = load16(xp[i] + kx);
    }
  };
  Split ws[TA];
  auto put = [&](int r, int k, int b) __attribute__((always_inline)) {
    if (k + SPLIT_BK > ke) {                               // columns past the end are zeros in both
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int a = 0; a < TA; ++a)
          if (k + 16 * h + 4 * lg >= ke) wr[r][a][h].u = zero16();
#pragma unroll
        for (int i = 0; i < EACH; ++i)
          if (k + 16 * h + 4 * xlg >= ke) xr[r][i][h].u = zero16();
      }
    }
#pragma unroll
    for (int a = 0; a < TA; ++a) ws[a] = split8(wr[r][a][0], wr[r][a][1]);
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      const Split s = split8(xr[r][i][0], xr[r][i][1]);
      uint4* at = lds + b * 3 * PIECES + split_piece(xrow + 64 * i, xlg);
      at[0] = s.h.u;
      at[PIECES] = s.m.u;
      at[2 * PIECES] = s.l.u;
    }
  };
  auto meet = [&]() __attribute__((always_inline)) {       // LDS is written and read; loads from memory stay under way
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  fetch(0, kb);
  fetch(1, kb + SPLIT_BK);
  put(0, kb, 0);
  __builtin_amdgcn_sched_barrier(0);
  fetch(0, kb + 2 * SPLIT_BK);
  meet();
  // the block at k from buffer b; that behind it is in registers 1 - b
  auto block = [&](int k, int b) __attribute__((always_inline)) {
    const uint4* xs = lds + b * 3 * PIECES;
    Split x[2];                                            // of 16 rows, and of the next
    auto read = [&](Split& to, int c) __attribute__((always_inline)) {
      const uint4* at = xs + split_piece(16 * c + ln, lg);
      to.h.u = at[0];
      to.m.u = at[PIECES];
      to.l.u = at[2 * PIECES];
    };
    read(x[0], 0);
#pragma unroll
    for (int c = 0; c < TC; ++c) {
      if (c >= groups) break;
      if (c + 1 < TC) read(x[(c + 1) & 1], c + 1);
      f32x4_t t[TA];
#pragma unroll
      for (int a = 0; a < TA; ++a) t[a] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#define STEP(S) _Pragma("unroll") for (int a = 0; a < TA; ++a) t[a] = split_step<S>(ws[a], x[c & 1], t[a]);
      STEP(0) STEP(1) STEP(2) STEP(3) STEP(4) STEP(5)
#undef STEP
#pragma unroll
      for (int a = 0; a < TA; ++a)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[a][c][i] += t[a][i];
      __builtin_amdgcn_sched_barrier(0);                   // (or all of x is read at once, into registers that are not there)
    }
    if (k + SPLIT_BK >= ke || (k + SPLIT_BK) % width == 0) done(k);
    put(1 - b, k + SPLIT_BK, 1 - b);                       // (behind the last block: zeros that nobody reads)
    __builtin_amdgcn_sched_barrier(0);                     // (the loads take the registers that have just become free)
    fetch(1 - b, k + 3 * SPLIT_BK);
    meet();
  };
  for (int k = kb; k < ke; k += 2 * SPLIT_BK) {
    block(k, 0);
    if (k + SPLIT_BK < ke) block(k + SPLIT_BK, 1);
  }
}
