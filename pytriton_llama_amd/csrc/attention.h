// What the attention kernels share beside their tables: which keys a query sees, and what is done
// to a row's result.
//
// A query at position p sees the keys at positions j <= p for which
//   window > 0   p - j < window (its own key and the window - 1 before it), or j < keep_first
//   chunk > 0    j / chunk == p / chunk (chunks of so many positions, counted from position 0)
//   neither      all of them
// (window and chunk exclude each other; keep_first goes with a window).
//
// sink (or null): one float a query head; the softmax denominator of that head holds exp(sink) once
// more, a term without key and value that is not scaled. gate (or null): one float a row and query
// head (row * gate_stride + head); the head's result is multiplied by sigmoid(gate).
//
// softcap > 0: a scaled score s becomes softcap * tanh(s / softcap) before the mask and the softmax.
#pragma once
#include "common.h"
#include <math.h>

struct AttnExtras {
  int window, keep_first, chunk;
  const float* sink;
  const float* gate;
  long gate_stride;
  float softcap;
};

// The first key that a query at position pos sees (of the window, for a window that keeps the
// sequence's first keys as well).
__device__ __forceinline__ int first_seen(const AttnExtras& ex, int pos) {
  if (ex.window > 0) return max(0, pos - ex.window + 1);
  if (ex.chunk > 0) return max(0, pos) / ex.chunk * ex.chunk;
  return 0;
}

// keys that the sequence's query reads (of the walk: the kept first keys, then the window)
__device__ __forceinline__ int walk_of(const AttnExtras& ex, int ctx) {
  const int lo = first_seen(ex, ctx - 1);
  return ctx - lo + min(max(ex.keep_first, 0), lo);
}
// keys of a split, a multiple of ``tile``
__device__ __forceinline__ int keys_a_split(int span, int num_splits, int tile) {
  return max(1, ((span + num_splits - 1) / num_splits + tile - 1) / tile) * tile;
}

__device__ __forceinline__ float head_gate(const AttnExtras& ex, int row, int head) {
  return ex.gate ? 1.0f / (1.0f + expf(-ex.gate[(size_t)row * ex.gate_stride + head])) : 1.0f;
}

__device__ __forceinline__ float cap_score(const AttnExtras& ex, float s) {
  return ex.softcap > 0.f ? ex.softcap * tanhf(s / ex.softcap) : s;
}

// tanh from the hardware's exp2 and reciprocal: 1 - 2 / (1 + e^(2x)), with x2 = 2 x log2 e. Absolute
// error of a few 1e-7 (the result feeds the exponent of a softmax); saturates to -1 and 1.
__device__ __forceinline__ float tanh_exp2(float x2) {
  return fmaf(-2.0f, __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x2)), 1.0f);
}

// Memory that another workgroup of the launch has written or will read.
__device__ __forceinline__ void put_shared(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float get_shared(const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// two of them, 8-byte aligned
__device__ __forceinline__ float2 get_shared2(const float* p) {
  return __builtin_bit_cast(float2, __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT));
}
// Workgroups that share a (sequence, kv head) pair's keys count in a ticket who is done. Tickets lie 16 bytes apart: those of one
// line are counted one after the other (one sequence, 8 pairs of 16 parts: 8.8 us side by side, 8.1 so and as 128 bytes apart).
constexpr int TICKET = 4;
// One more part of a pair is done (its writes have reached memory): whether it was the last one. The counter is zero again then.
__device__ __forceinline__ bool last_part(int* ticket, int parts) {
  const bool last = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == parts - 1;
  if (last) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return last;
}

static inline bool extras_ok(const AttnExtras& ex) {
  return ex.softcap >= 0.f && !(ex.chunk > 0 && (ex.window > 0 || ex.keep_first > 0));
}
