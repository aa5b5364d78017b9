// Tiles of float32 products on the matrix cores, shared by the kernels for dense matrices and for
// experts.
//
// v_mfma_f32_32x32x2_f32: lane l (r = l % 32, h = l / 32) holds A[r][k = h] and B[k = h][r] and gets
// D[8 (i / 4) + 4 h + i % 4][r], i = 0..15; float32 products and sums. Which k a lane holds is free as
// long as A and B agree, so a lane reads four consecutive floats of its row at once and hands them to
// four instructions.
//
// A step of F32_BK columns lies in LDS as rows of 32 floats, unpadded, the 16-byte pieces of a row
// permuted by (row / 2) % 8: eight neighbouring lanes touch all banks once, writing along a row and
// reading down a column of pieces alike.
#pragma once
#include <hip/hip_runtime.h>

typedef float f32x16_t __attribute__((ext_vector_type(16)));

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
