// Register types of the float32 kernels on the matrix cores.
//
// v_mfma_f32_16x16x4_f32: lane l (ln = l % 16, lg = l / 16) holds A[ln][k = lg] and B[k = lg][ln] and gets
// D[4 lg + i][ln], i = 0..3; float32 products and sums. Which k a lane holds is free as long as A and B agree, so a lane
// reads four consecutive floats of its row at once and hands them to four instructions.
#pragma once
#include <hip/hip_runtime.h>

typedef float f32x4_t __attribute__((ext_vector_type(4)));

union F4 {
  uint4 u;
  float f[4];
};
