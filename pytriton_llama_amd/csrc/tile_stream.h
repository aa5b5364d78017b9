// Rows of two matrices on their way through LDS, for products in which both are multiplied from there (gemm_tile.hip).
//
// A chunk is 128 bytes of every row of a tile (64 columns of bfloat16). Chunks lie in NB buffers; waves
// that do nothing else bring them, with loads that go from global memory to LDS without a register, NB - 1
// chunks ahead of the waves that multiply, and run on into the workgroup's next tile while the others store the results
// of this one. Two reasons for waves of their own. A weight comes from HBM, some 2 us away under load: a workgroup that loaded the
// next chunk while it multiplied one (0.2 to 0.5 us) waited for most of that. And the compiler lets no wave read LDS while a
// load to LDS is under way that might be of the same buffer, so a wave that did both could never have more than one
// chunk in flight.
//
// A load instruction fills 8 rows of 128 bytes, lane l the l-th 16 bytes: row l / 8, place l % 8, which holds the row's
// piece (l % 8) ^ (row % 8). A fragment read (16 neighbouring rows, the same piece, at piece ^ (row % 8)) then meets no bank
// twice (counted: no conflicts). One such wave issues a load every 66 to 83 clocks, 12 to 15 bytes a clock of the 50
// that a compute unit takes from L2: hence four of them, one beside every wave that multiplies (gemm_tile.hip, us with two
// and with four: 277 x 16,384 x 2,048 28.7 / 27.8, 277 x 2,048 x 8,192 19.2 / 18.6, 532 x 16,384 x 3,072 56.1 / 54.2, 1,000 x 16,384 x
// 2,048 71.2 / 69.4; a group of 8 rows more for some of them where four do not share a tile's evenly).
#pragma once
#include <hip/hip_runtime.h>

constexpr int TILE_ROW = 128;                    // bytes of a row in a chunk

// All waves of the workgroup meet; nothing but the meeting (the loads a wave has under way
// stay under way). The clobbers keep the compiler from moving LDS accesses across it.
__device__ __forceinline__ void tile_meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// s_waitcnt vmcnt(N) alone (expcnt and lgkmcnt left at their maxima)
template <int N> __device__ __forceinline__ void tile_wait_loads_but() {
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// s_waitcnt lgkmcnt(0): what the wave has read from LDS is in its registers
__device__ __forceinline__ void tile_wait_lds() { __builtin_amdgcn_s_waitcnt(0xC07F); }

// What a loading wave does that brings LI groups of 8 rows, from the ``first`` on.
template <int ROWS, int NB, int LI, typename Rows>
__device__ __forceinline__ void tile_bring_groups(unsigned char* lds, int first, int lane, int tiles, int chunks, Rows rows) {
  static_assert(NB >= 3 && NB <= 5 && (NB - 2) * LI < 64, "loads are counted in six bits");
  const int lrow = lane >> 3, lpiece = (lane & 7) ^ lrow;
  const char* src[LI];
  int next = 0, next_tile = 0, next_chunk = 0, slot = 0;
  const int all = tiles * chunks;
  auto fetch = [&]() __attribute__((always_inline)) {
    if (next_chunk == 0) {
#pragma unroll
      for (int i = 0; i < LI; ++i) src[i] = rows(next_tile, 8 * (first + i) + lrow) + 16 * lpiece;
    }
    unsigned char* dst = lds + (size_t)slot * (ROWS * TILE_ROW) + 1024 * first;
#pragma unroll
    for (int i = 0; i < LI; ++i) {
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src[i],
                                       (__attribute__((address_space(3))) void*)(dst + 1024 * i), 16, 0, 0);
      src[i] += TILE_ROW;
    }
    ++next;
    slot = slot + 1 == NB ? 0 : slot + 1;
    if (++next_chunk == chunks) { next_chunk = 0; ++next_tile; }
  };
  for (int c = 0; c < NB - 1; ++c)
    if (next < all) fetch();
  for (int c = 0; c < all; ++c) {
    // chunk c has landed when at most the chunks after it are still under way
    switch (min(NB - 2, all - 1 - c)) {
      case 0: tile_wait_loads_but<0>(); break;
      case 1: tile_wait_loads_but<LI>(); break;
      case 2: tile_wait_loads_but<(NB > 3 ? 2 * LI : 0)>(); break;
      default: tile_wait_loads_but<(NB > 4 ? 3 * LI : 0)>(); break;
    }
    tile_meet();                                 // chunk c is there; chunk c - 1 has been read
    if (next < all) fetch();
  }
}

// What a loading wave does (``me``: which of the PW): ``tiles`` tiles of ROWS rows one after the other, ``chunks`` chunks
// each. rows(i, r): where row r of the workgroup's i-th tile begins (a valid row for every r < ROWS), in bytes, at
// the first column the tile takes. The other waves call tile_meet() once a chunk before they read it, in the same order.
template <int ROWS, int NB, int PW, typename Rows>
__device__ __forceinline__ void tile_bring(unsigned char* lds, int me, int lane, int tiles, int chunks, Rows rows) {
  static_assert(ROWS % 8 == 0 && ROWS / 8 >= PW, "groups of 8 rows");
  constexpr int EACH = ROWS / 8 / PW, MORE = ROWS / 8 % PW;    // (the first MORE waves bring one more)
  if (MORE > 0 && me < MORE) tile_bring_groups<ROWS, NB, EACH + 1>(lds, me * (EACH + 1), lane, tiles, chunks, rows);
  else tile_bring_groups<ROWS, NB, EACH>(lds, me * EACH + MORE, lane, tiles, chunks, rows);
}

// The order of a stage of R reads from LDS (for the next stage) and P matrix instructions: the reads one at a time
// within the first three quarters of the products. Issued together they hold the wave's products up until LDS
// has taken the last of them (2,048 x 2,048 x 8,192 in bfloat16, tiles of 128 x 128: 68 us together, 58 so).
template <int R, int P> __device__ __forceinline__ void tile_interleave() {
  constexpr int EACH = P * 3 / (4 * R) > 0 ? P * 3 / (4 * R) : 1;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);       // one read of LDS
    __builtin_amdgcn_sched_group_barrier(0x008, EACH, 0);    // some matrix instructions
  }
  if (P > EACH * R) __builtin_amdgcn_sched_group_barrier(0x008, P - EACH * R, 0);
  __builtin_amdgcn_sched_barrier(0);
}
