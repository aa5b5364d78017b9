// Tiles of float32 products on the matrix cores, for dense matrices (f32_multiply16) and for experts
// (f32_multiply).
//
// v_mfma_f32_32x32x2_f32: lane l (r = l % 32, h = l / 32) holds A[r][k = h] and B[k = h][r] and gets
// D[8 (i / 4) + 4 h + i % 4][r], i = 0..15; float32 products and sums. Which k a lane holds is free as
// long as A and B agree, so a lane reads four consecutive floats of its row at once and hands them to
// four instructions. v_mfma_f32_16x16x4_f32, at the same rate: lane l (ln = l % 16, lg = l / 16) holds
// A[ln][k = lg] and B[k = lg][ln] and gets D[4 lg + i][ln], i = 0..3.
//
// A step of F32_BK columns lies in LDS as rows of 32 floats, unpadded, the 16-byte pieces of a row
// permuted by (row / 2) % 8: eight neighbouring lanes touch all banks once, writing along a row and
// reading down a column of pieces alike.
#pragma once
#include <hip/hip_runtime.h>

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

#define F32_BK 32

union F4 {
  uint4 u;
  float f[4];
};

__device__ __forceinline__ int f32_piece(int row, int piece) { return row * 8 + (piece ^ ((row >> 1) & 7)); }

// acc[a][b] += A rows (arow[a] .. + 31) x B rows (brow[b] .. + 31)^T over the F32_BK columns in As and Bs:
// for 8 columns a wave reads TA + TB fragments and issues 4 TA TB instructions of 64 clocks.
template <int TA, int TB>
__device__ __forceinline__ void f32_multiply(f32x16_t (&acc)[TA][TB], const uint4* As, const uint4* Bs,
                                             const int (&arow)[TA], const int (&brow)[TB], int lane) {
  const int r = lane & 31, h = lane >> 5;
  F4 fa[2][TA], fb[2][TB];
#pragma unroll
  for (int a = 0; a < TA; ++a) fa[0][a].u = As[f32_piece(arow[a] + r, h)];
#pragma unroll
  for (int b = 0; b < TB; ++b) fb[0][b].u = Bs[f32_piece(brow[b] + r, h)];
#pragma unroll
  for (int g = 0; g < F32_BK / 8; ++g) {
    if (g + 1 < F32_BK / 8) {
#pragma unroll
      for (int a = 0; a < TA; ++a) fa[(g + 1) & 1][a].u = As[f32_piece(arow[a] + r, 2 * (g + 1) + h)];
#pragma unroll
      for (int b = 0; b < TB; ++b) fb[(g + 1) & 1][b].u = Bs[f32_piece(brow[b] + r, 2 * (g + 1) + h)];
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int a = 0; a < TA; ++a)
#pragma unroll
        for (int b = 0; b < TB; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[g & 1][a].f[s], fb[g & 1][b].f[s], acc[a][b], 0, 0, 0);
  }
}

// acc[block % 2][a][b] += A rows (a_row + 16 a ..) x B rows (b_row + 16 b ..)^T over the blocks of 16 columns in As and
// Bs (F32_BK in all), instruction s of a block columns 3 - s, 7 - s, 11 - s and 15 - s: for a block a wave reads
// TA + TB fragments and issues 4 TA TB instructions of 32 clocks.
template <int TA, int TB>
__device__ __forceinline__ void f32_multiply16(f32x4_t (&acc)[2][TA][TB], const uint4* As, const uint4* Bs, int a_row,
                                               int b_row, int lane) {
  static_assert(F32_BK == 32, "an even and an odd block");
  const int ln = lane & 15, lg = lane >> 4;
  F4 fa[2][TA], fb[2][TB];
#pragma unroll
  for (int g = 0; g < 2; ++g) {
#pragma unroll
    for (int a = 0; a < TA; ++a) fa[g][a].u = As[f32_piece(a_row + 16 * a + ln, 4 * g + lg)];
#pragma unroll
    for (int b = 0; b < TB; ++b) fb[g][b].u = Bs[f32_piece(b_row + 16 * b + ln, 4 * g + lg)];
  }
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int a = 0; a < TA; ++a)
#pragma unroll
        for (int b = 0; b < TB; ++b)
          acc[g][a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[g][a].f[3 - s], fb[g][b].f[3 - s], acc[g][a][b], 0, 0, 0);
}
