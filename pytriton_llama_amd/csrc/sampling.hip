// Sampling from float32 logits [R, V], one workgroup per row.
//
// ptl_argmax: greedy choice, ties to the lowest id (the reference's greedy
// branch is torch.argmax, lite_llama/generate_stream.py:150).
//
// ptl_sample_top_p: softmax(logits / temperature) (the reference's three-pass
// split softmax, lite_llama/kernels/softmax_split.py:7-77) followed by nucleus
// sampling with the rule of lite_llama/generate.py:30-43: in descending order of
// probability a token is kept while the mass before it is <= top_p, the kept
// ones are renormalised and one is drawn. The draw uses a uniform number
// u[r] in [0,1) given by the caller (seeded per request and step on the host),
// so a result does not depend on what else is in the batch.
//
// Instead of a sort the kernel finds the smallest kept probability by bisection
// over float bit patterns: mass_above(t) = sum of p > t never grows with t, and
// a token of probability p is kept iff mass_above(p) <= top_p. Tokens of equal
// probability are kept or dropped together; a sort would split such a tie at
// the edge of the nucleus by index.
#include "common.h"
#include "no_alloc.h"
#include <math.h>
#include <string.h>
#include <mutex>

// Two passes so that a row of vocabulary size is read by many workgroups: every
// chunk leaves its best (value, index), then one wave per row picks among them.
#define ARGMAX_CHUNK 4096

__device__ __forceinline__ void argmax_pick(float& best, int& bi, float v, int i) {
  if (v > best || (v == best && i < bi)) { best = v; bi = i; }
}

__global__ void __launch_bounds__(256)
argmax_partial_kernel(float* __restrict__ pv, int32_t* __restrict__ pi,
                      const float* __restrict__ logits, int V, long stride, int chunks) {
  __shared__ float sv[4];
  __shared__ int si[4];
  const float* row = logits + (size_t)blockIdx.y * stride;
  const int lo = blockIdx.x * ARGMAX_CHUNK, hi = min(V, lo + ARGMAX_CHUNK);
  float best = -INFINITY;
  int bi = 0x7fffffff;
  if (hi - lo == ARGMAX_CHUNK && (reinterpret_cast<uintptr_t>(row + lo) & 15) == 0) {
    // a whole chunk with 16-byte aligned rows: a thread's four loads are asked for at once
    float4 v[ARGMAX_CHUNK / 1024];
#pragma unroll
    for (int k = 0; k < ARGMAX_CHUNK / 1024; ++k)
      v[k] = *reinterpret_cast<const float4*>(row + lo + 4 * (threadIdx.x + 256 * k));
#pragma unroll
    for (int k = 0; k < ARGMAX_CHUNK / 1024; ++k) {
      const float e[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
#pragma unroll
      for (int j = 0; j < 4; ++j)
        argmax_pick(best, bi, e[j] != e[j] ? -INFINITY : e[j], lo + 4 * (threadIdx.x + 256 * k) + j);
    }
  } else {
    for (int i = lo + threadIdx.x; i < hi; i += 256) {
      float v = row[i];
      if (v != v) v = -INFINITY;
      argmax_pick(best, bi, v, i);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) argmax_pick(best, bi, __shfl_xor(best, o, 64), __shfl_xor(bi, o, 64));
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 0) { sv[wave] = best; si[wave] = bi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < 4; ++i) argmax_pick(best, bi, sv[i], si[i]);
    pv[(size_t)blockIdx.y * chunks + blockIdx.x] = best;
    pi[(size_t)blockIdx.y * chunks + blockIdx.x] = bi;
  }
}

// host_out (optional): pinned host memory that receives the choices as well, written over the
// bus by this kernel, so that the host needs no copy after it
__global__ void __launch_bounds__(64)
argmax_final_kernel(int32_t* __restrict__ out, const float* __restrict__ pv,
                    const int32_t* __restrict__ pi, int chunks, int32_t* __restrict__ host_out) {
  float best = -INFINITY;
  int bi = 0x7fffffff;
  for (int i = threadIdx.x; i < chunks; i += 64)
    argmax_pick(best, bi, pv[(size_t)blockIdx.x * chunks + i], pi[(size_t)blockIdx.x * chunks + i]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) argmax_pick(best, bi, __shfl_xor(best, o, 64), __shfl_xor(bi, o, 64));
  if (threadIdx.x == 0) {
    const int choice = bi == 0x7fffffff ? 0 : bi;
    out[blockIdx.x] = choice;
    if (host_out != nullptr) host_out[blockIdx.x] = choice;
  }
}

// workspace: float [R, chunks] and int32 [R, chunks], chunks = ceil(V / 4096)
extern "C" int ptl_argmax(int32_t* out, const float* logits, int R, int V, long stride,
                          float* ws_val, int32_t* ws_idx, int32_t* host_out, hipStream_t stream) {
  if (R <= 0) return PTL_OK;
  if (V <= 0 || stride < V || !ws_val || !ws_idx || R > 65535) return PTL_ERR_ARG;
  const int chunks = (V + ARGMAX_CHUNK - 1) / ARGMAX_CHUNK;
  dim3 grid(chunks, R);
  argmax_partial_kernel<<<grid, 256, 0, stream>>>(ws_val, ws_idx, logits, V, stride, chunks);
  if (hipGetLastError() != hipSuccess) return PTL_ERR_LAUNCH;
  argmax_final_kernel<<<R, 64, 0, stream>>>(out, ws_val, ws_idx, chunks, host_out);
  return ptl_launch_status();
}

// ptl_argmax with its workspace inside the library (see no_alloc.h): values in the first half of
// the array, indices in the second. Host code never uses the array's name as an address: the
// name is a host-side stand-in; the device address comes from hipGetSymbolAddress, once per
// device with that device current (every GPU holds a copy of its own), and is what the
// kernels are given.
static __device__ __align__(256) unsigned char argmax_scratch[PTL_ARGMAX_STATIC_MAX_PARTIALS * 8];
#define ARGMAX_STATIC_MAX_DEVICES 64
static void* argmax_scratch_at[ARGMAX_STATIC_MAX_DEVICES];
static std::mutex argmax_scratch_lock;

// The array's address on device ``dev``, looked up the first time with that device current.
// ``may_look_up`` false: only what is known already (a look-up may load the code object onto the
// device, which is no work for a stream that is being captured).
static int argmax_scratch_of(int dev, bool may_look_up, void** base) {
  if (dev < 0 || dev >= ARGMAX_STATIC_MAX_DEVICES) return PTL_ERR_LAUNCH;
  std::lock_guard<std::mutex> hold(argmax_scratch_lock);
  if (argmax_scratch_at[dev] == nullptr) {
    if (!may_look_up) return PTL_ERR_LAUNCH;
    int current = -1;
    if (hipGetDevice(&current) != hipSuccess) {
      (void)hipGetLastError();
      return PTL_ERR_LAUNCH;
    }
    if (current != dev && hipSetDevice(dev) != hipSuccess) {
      (void)hipGetLastError();
      return PTL_ERR_LAUNCH;
    }
    void* p = nullptr;
    const hipError_t found = hipGetSymbolAddress(&p, HIP_SYMBOL(argmax_scratch));
    if (current != dev) (void)hipSetDevice(current);
    if (found != hipSuccess || p == nullptr) {
      (void)hipGetLastError();
      return PTL_ERR_LAUNCH;
    }
    argmax_scratch_at[dev] = p;
  }
  *base = argmax_scratch_at[dev];
  return PTL_OK;
}

// The device a stream belongs to (the current device for the null stream).
static int device_of(hipStream_t stream) {
  int dev = -1;
  if (stream != nullptr && hipStreamGetDevice(stream, &dev) == hipSuccess) return dev;
  (void)hipGetLastError();
  if (hipGetDevice(&dev) != hipSuccess) {
    (void)hipGetLastError();
    return -1;
  }
  return dev;
}

extern "C" int ptl_argmax_static_init(void) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess) {
    (void)hipGetLastError();
    return PTL_ERR_LAUNCH;
  }
  void* base = nullptr;
  return argmax_scratch_of(dev, true, &base);
}

extern "C" int ptl_argmax_static(int32_t* out, const float* logits, int R, int V, long stride,
                                 int32_t* host_out, hipStream_t stream) {
  if (R <= 0) return PTL_OK;
  if (!out || !logits || V <= 0 || stride < V || R > 65535) return PTL_ERR_ARG;
  const long chunks = ((long)V + ARGMAX_CHUNK - 1) / ARGMAX_CHUNK;
  if ((long)R * chunks > PTL_ARGMAX_STATIC_MAX_PARTIALS) return PTL_ERR_ARG;
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &capturing) != hipSuccess) {
    (void)hipGetLastError();
    capturing = hipStreamCaptureStatusNone;
  }
  void* base = nullptr;
  const int rc = argmax_scratch_of(device_of(stream), capturing == hipStreamCaptureStatusNone, &base);
  if (rc != PTL_OK) return rc;
  float* ws_val = reinterpret_cast<float*>(base);
  int32_t* ws_idx = reinterpret_cast<int32_t*>(static_cast<unsigned char*>(base) +
                                               (size_t)PTL_ARGMAX_STATIC_MAX_PARTIALS * 4);
  return ptl_argmax(out, logits, R, V, stride, ws_val, ws_idx, host_out, stream);
}

// probs_out (optional, [R, V]) receives the renormalised nucleus distribution.
//
// How the nucleus is found without a sort. With e = exp(logit/T - max) (the unnormalised
// probability, kept in the work buffer), a token is kept iff the mass of the tokens with
// larger e is <= top_p * sum(e).
// (1) row max; (2) e and its sum; (3) three rounds of a 16-way split of the distance from
// the max, d = -ln e: round one splits [0, 32) into 16 buckets, finds the bucket in which
// the cumulative mass (most likely tokens first) crosses top_p, and the next rounds split
// that bucket again, down to a width of 1/128. Every thread adds into a column of its own
// in LDS (no atomics: LDS float atomics cost about a hundred cycles a wave here); (4) the
// tokens of the last crossing bucket (a few dozen for ordinary logits) are gathered and the
// exact cut among them is found by one wave bisecting over float bit patterns, ending with
// two neighbouring floats so that no e lies between them; (5) the waves sum their kept mass
// over contiguous ranges, a scan locates the wave whose range holds u * kept, and that wave
// walks its range with a running prefix. If the last bucket holds more tokens than fit (many
// equal logits), the bisection runs over the whole row: slower, same result.
#define SMP_THREADS 1024
#define SMP_FAN 16               // buckets per round
#define SMP_ROUNDS 3
#define SMP_SPAN 32.0f           // distance from the max that round one covers
#define SMP_LIST 4096

// exclusive prefix sum over the block; tmp holds 17 floats. Returns the prefix, total in *total.
__device__ __forceinline__ float block_exclusive_scan(float v, float* tmp, float* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  float inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float n = __shfl_up(inc, o, 64);
    if (lane >= o) inc += n;
  }
  __syncthreads();
  if (lane == 63) tmp[wave] = inc;
  __syncthreads();
  if (threadIdx.x == 0) {
    float run = 0.f;
    for (int i = 0; i < nw; ++i) { const float t = tmp[i]; tmp[i] = run; run += t; }
    tmp[16] = run;
  }
  __syncthreads();
  *total = tmp[16];
  return tmp[wave] + inc - v;
}

// Every pass over a row: four consecutive values a thread and step (one 16-byte load) when the
// row is 16-byte aligned, then the few values that are left; f(i, value).
template <typename F>
__device__ __forceinline__ void for_row(const float* __restrict__ p, int V, bool vec, F f) {
  if (vec) {
    // (four loads under way at a time: a pass is a chain of L2 round trips otherwise)
    const int n4 = V >> 2;
    const int step = blockDim.x;
    const float4* p4 = reinterpret_cast<const float4*>(p);
    int i = threadIdx.x;
    for (; i + 3 * step < n4; i += 4 * step) {
      float4 v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = p4[i + j * step];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int at = 4 * (i + j * step);
        f(at, v[j].x); f(at + 1, v[j].y); f(at + 2, v[j].z); f(at + 3, v[j].w);
      }
    }
    for (; i < n4; i += step) {
      const float4 v = p4[i];
      f(4 * i, v.x); f(4 * i + 1, v.y); f(4 * i + 2, v.z); f(4 * i + 3, v.w);
    }
    for (int t = 4 * n4 + threadIdx.x; t < V; t += step) f(t, p[t]);
  } else {
    for (int i = threadIdx.x; i < V; i += blockDim.x) f(i, p[i]);
  }
}

// work: float [R, V] scratch of the caller; it receives exp(logit/T - max) in the second
// pass, which the later passes read back instead of computing it again, and in the end (if
// want_probs) the renormalised nucleus distribution.
__global__ void __launch_bounds__(SMP_THREADS)
sample_top_p_kernel(int32_t* __restrict__ out, float* __restrict__ work, int want_probs,
                    const float* __restrict__ logits, int V, long stride,
                    const float* __restrict__ temperature, const float* __restrict__ top_p,
                    const float* __restrict__ uniform) {
  __shared__ float scratch[17];
  __shared__ float cols[SMP_FAN * SMP_THREADS];      // a column of bucket sums per thread
  __shared__ float part[SMP_FAN * 16];
  __shared__ float bucket[SMP_FAN];
  __shared__ float list[SMP_LIST];
  __shared__ int list_n;
  __shared__ int cross_bin;
  __shared__ float mass_before;
  __shared__ float thr_s;
  __shared__ int last_kept;
  const int tid = threadIdx.x;
  const int r = blockIdx.x;
  const float* row = logits + (size_t)r * stride;
  float* ex = work + (size_t)r * V;          // unnormalised probabilities e_i = exp(x_i/T - max)
  const float inv_t = 1.0f / temperature[r];
  const float c = inv_t * 1.4426950408889634f;

  const bool vec_in = (((uintptr_t)row) & 15) == 0, vec_ex = (((uintptr_t)ex) & 15) == 0;
  float mx = -INFINITY;
  for_row(row, V, vec_in, [&](int, float x) { mx = fmaxf(mx, x); });
  mx = block_max(mx, scratch);
  const float mc = mx * c;
  float z = 0.f;
  // (a NaN logit counts as -inf: probability 0)
  float emax = 0.f;                          // the largest e (1 up to rounding)
  auto expo = [&](float x) {
    const float e = x != x ? 0.f : __builtin_amdgcn_exp2f(fmaf(x, c, -mc));
    emax = fmaxf(emax, e);
    return e;
  };
  if (vec_in && vec_ex) {
    const int n4 = V >> 2;
    auto exp4 = [&](int i, float4 x) {
      float4 e;
      e.x = expo(x.x);
      e.y = expo(x.y);
      e.z = expo(x.z);
      e.w = expo(x.w);
      reinterpret_cast<float4*>(ex)[i] = e;
      z += (e.x + e.y) + (e.z + e.w);
    };
    int i = tid;
    for (; i + 3 * SMP_THREADS < n4; i += 4 * SMP_THREADS) {
      float4 x[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = reinterpret_cast<const float4*>(row)[i + j * SMP_THREADS];
#pragma unroll
      for (int j = 0; j < 4; ++j) exp4(i + j * SMP_THREADS, x[j]);
    }
    for (; i < n4; i += SMP_THREADS) exp4(i, reinterpret_cast<const float4*>(row)[i]);
    for (int i = 4 * n4 + tid; i < V; i += SMP_THREADS) {
      const float e = expo(row[i]);
      ex[i] = e;
      z += e;
    }
  } else {
    for (int i = tid; i < V; i += SMP_THREADS) {
      const float e = expo(row[i]);
      ex[i] = e;
      z += e;
    }
  }
  z = block_sum(z, scratch);                 // (its barriers also publish ex[] to the block)
  emax = block_max(emax, scratch);
  const float tp = top_p[r] * z;             // all masses below are in units of e
  float thr = -1.0f;                         // kept: e > thr
  if (top_p[r] < 1.0f) {
    // Round q splits [lo[q], lo[q] + SMP_FAN / inv_w[q]) of d = -ln e into SMP_FAN buckets and
    // picks bucket pick[q]. A token belongs to a later round (and to the final list) iff the
    // same arithmetic put it into the picked bucket of every earlier round, so that no token
    // near a bucket's edge is counted twice or lost.
    float lo[SMP_ROUNDS], inv_w[SMP_ROUNDS];
    int pick[SMP_ROUNDS];
    float lo_d = 0.f, width = SMP_SPAN / SMP_FAN;
    float mb = 0.f;                          // mass of everything more likely than the bucket in hand
    bool found = true;
    if (tid == 0) list_n = 0;
    auto bucket_of = [&](float d, int q) -> int {
      float fb = (d - lo[q]) * inv_w[q];
      if (q == 0) fb = fminf(fmaxf(fb, 0.f), (float)(SMP_FAN - 1));   // far tokens: last bucket
      return (fb >= 0.f && fb < (float)SMP_FAN) ? (int)fb : -1;
    };
#pragma unroll
    for (int round = 0; round < SMP_ROUNDS; ++round) {
      if (!found) break;
      lo[round] = lo_d;
      inv_w[round] = 1.0f / width;
      for (int b = 0; b < SMP_FAN; ++b) cols[b * SMP_THREADS + tid] = 0.f;
      for_row(ex, V, vec_ex, [&](int, float e) {
        const float d = fmaxf(-__builtin_amdgcn_logf(e) * 0.6931471805599453f, 0.f);   // e may be a hair above 1
        bool in = true;
#pragma unroll
        for (int q = 0; q < round; ++q) in = in && bucket_of(d, q) == pick[q];
        const int bk = bucket_of(d, round);
        if (in && bk >= 0) cols[bk * SMP_THREADS + tid] += e;
      });
      // bucket sums: wave sums, then sixteen threads add the waves' partial sums
      for (int b = 0; b < SMP_FAN; ++b) {
        const float v = wave_sum(cols[b * SMP_THREADS + tid]);
        if ((tid & 63) == 0) part[b * 16 + (tid >> 6)] = v;
      }
      __syncthreads();
      if (tid < SMP_FAN) {
        float v = 0.f;
        for (int w = 0; w < 16; ++w) v += part[tid * 16 + w];
        bucket[tid] = v;
      }
      __syncthreads();
      if (tid == 0) {
        float run = mb;
        int cb = -1;
        for (int b = 0; b < SMP_FAN; ++b) {
          if (run + bucket[b] > tp) { cb = b; break; }
          run += bucket[b];
        }
        cross_bin = cb;
        mass_before = run;
      }
      __syncthreads();
      pick[round] = cross_bin;
      mb = mass_before;
      if (pick[round] < 0) { found = false; break; }   // rounding left the whole mass <= top_p
      lo_d += pick[round] * width;
      width *= 1.0f / SMP_FAN;
    }
    if (found) {
      for_row(ex, V, vec_ex, [&](int, float e) {
        const float d = fmaxf(-__builtin_amdgcn_logf(e) * 0.6931471805599453f, 0.f);   // e may be a hair above 1
        bool in = true;
#pragma unroll
        for (int q = 0; q < SMP_ROUNDS; ++q) in = in && bucket_of(d, q) == pick[q];
        if (in) {
          const int at = atomicAdd(&list_n, 1);
          if (at < SMP_LIST) list[at] = e;
        }
      });
      __syncthreads();
      const int n = list_n;
      // lo keeps mass_above(lo) > top_p, hi keeps mass_above(hi) <= top_p
      uint32_t lo = 0u, hi = __float_as_uint(2.0f);
      if (n <= SMP_LIST) {
        if (tid < 64) {                      // the list is short: one wave bisects it
          while (hi - lo > 1u) {
            const uint32_t mid = lo + ((hi - lo) >> 1);
            const float t = __uint_as_float(mid);
            float mass = 0.f;
            for (int i = tid; i < n; i += 64) mass += list[i] > t ? list[i] : 0.f;
            mass = wave_sum(mass) + mb;
            if (mass <= tp) hi = mid; else lo = mid;
          }
          if (tid == 0) thr_s = __uint_as_float(lo);
        }
        __syncthreads();
      } else {                               // too many tokens in one bucket: bisect over the whole row
        while (hi - lo > 1u) {
          const uint32_t mid = lo + ((hi - lo) >> 1);
          const float t = __uint_as_float(mid);
          float mass = 0.f;
          for (int i = tid; i < V; i += SMP_THREADS) {
            const float e = ex[i];
            if (e > t) mass += e;
          }
          mass = block_sum(mass, scratch);
          if (mass <= tp) hi = mid; else lo = mid;
        }
        if (tid == 0) thr_s = __uint_as_float(lo);
        __syncthreads();
      }
      thr = thr_s;
      // the most likely token is always kept: nothing lies before it
      if (thr >= emax) thr = __uint_as_float(__float_as_uint(emax) - 1u);
    }
  }

  // inverse-CDF draw in vocabulary order. Every wave owns a contiguous range and reads it
  // 64 tokens at a time (coalesced); the waves' kept masses are scanned, and the wave whose
  // range holds u * kept walks it again with a running prefix.
  const int lane = tid & 63, wave = tid >> 6;
  const int per_wave = ((V + 15) / 16 + 63) / 64 * 64;
  const int wb = wave * per_wave, we = min(V, wb + per_wave);
  float mine = 0.f;
  for (int i = wb + lane; i < we; i += 64) {
    const float e = ex[i];
    if (e > thr) mine += e;
  }
  mine = wave_sum(mine);
  float kept;
  const float before = block_exclusive_scan(lane == 0 ? mine : 0.f, scratch, &kept);
  const float wave_before = __shfl(before, 0, 64);
  const float target = uniform[r] * kept;
  if (tid == 0) { out[r] = -1; last_kept = 0; }
  __syncthreads();
  if (mine > 0.f) {
    const bool owner = wave_before <= target && target < wave_before + mine;
    float run = wave_before;
    int choice = -1, my_last = -1;
    for (int i0 = wb; i0 < we; i0 += 64 * 8) {
      float ev[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {           // eight loads in flight, then eight scans
        const int i = i0 + 64 * k + lane;
        ev[k] = (i < we) ? ex[i] : 0.f;
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int i = i0 + 64 * k + lane;
        const float v = ev[k] > thr ? ev[k] : 0.f;
        if (v > 0.f) my_last = i;
        if (owner && choice < 0) {
          float inc = v;
#pragma unroll
          for (int o = 1; o < 64; o <<= 1) {
            const float nb = __shfl_up(inc, o, 64);
            if (lane >= o) inc += nb;
          }
          const unsigned long long hit = __ballot(v > 0.f && run + inc > target);
          if (hit) choice = i0 + 64 * k + __ffsll((long long)hit) - 1;
          run += __shfl(inc, 63, 64);
        }
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) my_last = max(my_last, __shfl_xor(my_last, o, 64));
    if (lane == 0) {
      if (owner) out[r] = choice >= 0 ? choice : my_last;
      atomicMax(&last_kept, my_last);
    }
  }
  __syncthreads();
  // rounding may leave the target past the last kept token: take that token
  if (tid == 0 && out[r] < 0) out[r] = last_kept;
  if (want_probs) {
    const float inv_kept = 1.0f / kept;
    for (int i = tid; i < V; i += SMP_THREADS) {
      const float e = ex[i];
      ex[i] = e > thr ? e * inv_kept : 0.f;
    }
  }
#undef BIN
}

extern "C" int ptl_sample_top_p(int32_t* out, float* work, int want_probs, const float* logits, int R,
                                int V, long stride, const float* temperature, const float* top_p,
                                const float* uniform, hipStream_t stream) {
  if (R <= 0) return PTL_OK;
  if (V <= 0 || stride < V || !work) return PTL_ERR_ARG;
  sample_top_p_kernel<<<R, SMP_THREADS, 0, stream>>>(out, work, want_probs, logits, V, stride,
                                                     temperature, top_p, uniform);
  return ptl_launch_status();
}

// ===========================================================================
// ptl_sample_top_p_wide: the same rule for rows of vocabulary size, spread over the chip.
//
// One workgroup reads a row of 128k logits at a small part of what the chip can deliver, and
// the kernel above passes over the row seven times. Here a row is cut into chunks of 4096
// logits, a workgroup a chunk, and the passes become kernels:
//   (1) scan:    every chunk's largest and smallest finite logit, its sum of exp(x/T - chunk max), and the tokens that the
//                nucleus can be made of (below);
//       small:   one workgroup a row draws the token from these, if there are few, and the kernels that
//                follow leave at once: a model's logits are peaked, and 64 rows of 128,256 have some 300
//                candidates each. Not for rows with top_p 1 and not if the probabilities are asked for;
//   (2) hist:    the chunk's sum of e = exp(x/T - max) and its histogram of that mass over 2048
//                buckets of x, equally wide, from the row's max down to its min (at most 32 T
//                below the max; what lies further goes to the last bucket). The histogram is
//                summed in LDS in fixed point (2^-40) with integer atomics, so that it does not
//                depend on the order of the threads; the last bucket, where most of a
//                vocabulary lies, in a register of every thread first (all of a wave's lanes
//                adding to one address: 40 instead of 17 us for 64 rows of 128,256);
//   (3) combine: one workgroup a row adds the chunks' histograms in chunk order and finds the
//                bucket in which the mass, most likely tokens first, passes top_p;
//   (4) gather:  every workgroup adds up what its chunk has above that bucket and hands on its
//                tokens inside it (at most 256);
//   (5) draw:    one workgroup a row bisects over the bit patterns of x among the tokens handed
//                on (a few hundred) for the exact edge of the nucleus, adds the kept mass chunk
//                by chunk, finds the chunk that holds u * kept and walks it;
//   (6) probs:   only if asked for, the renormalised nucleus distribution.
// A token is kept iff it lies in a bucket above the crossing one, or in it and above the edge;
// equal logits are kept or dropped together. e is worked out again from x wherever it is wanted
// (one multiplication, one exp2, the same bits): keeping it would be a write and a read of the
// whole row. 64 rows of 128,256 logits (one MI355X): 66 us for the five kernels without small, 12 to 17 for each of the
// three passes over the logits, of which peaked rows take one: scan 13.6, small 12.6, the others 2 to 3 each, 35 us
// in all (rows with too many candidates 71); 97 us with e kept, the crossing found by every workgroup of the gather
// kernel and the last bucket in LDS. If a chunk has more than 256 tokens in the crossing
// bucket, or the row more than 4096 (many equal logits), the draw kernel bisects over the whole
// row instead: slower, same result. Everything is added in a fixed order: the same logits,
// parameters and u give the same token.
// ===========================================================================
#define SW_CHUNK 4096
#define SW_THREADS 256
#define SW_PER (SW_CHUNK / SW_THREADS)
#define SW_BUCKETS 2048
#define SW_SEG 256
#define SW_LIST 4096
#define SW_SPAN 32.0f
#define SW_FIXED 1099511627776.0f        // 2^40

// where a row's pieces lie in the workspace (all 4-byte words)
struct SwRow {
  float *cmax, *cmin, *csum, *ckept, *hist, *seg_x, *result;
  int32_t *ccount, *seg_i;
};
__host__ __device__ static inline size_t sw_row_words(int S) {
  return (size_t)5 * S + (size_t)S * SW_BUCKETS + (size_t)2 * S * SW_SEG + 12;
}
__device__ __forceinline__ SwRow sw_row(float* ws, int r, int S) {
  float* p = ws + (size_t)r * sw_row_words(S);
  SwRow w;
  w.cmax = p; p += S;
  w.cmin = p; p += S;
  w.csum = p; p += S;
  w.ckept = p; p += S;
  w.ccount = reinterpret_cast<int32_t*>(p); p += S;
  w.hist = p; p += (size_t)S * SW_BUCKETS;
  w.seg_x = p; p += (size_t)S * SW_SEG;
  w.seg_i = reinterpret_cast<int32_t*>(p); p += (size_t)S * SW_SEG;
  w.result = p;        // [0] edge key (bits), [1] crossing bucket (bits), [2] kept mass, [3] mass before
                       // the crossing bucket, [4] row max, [5] buckets per unit of x, [6] sum of e,
                       // [7] not 0: the token is drawn, [8] temperature, [9] top_p, [10] u
  return w;
}

// bit patterns that order as the floats do
__device__ __forceinline__ uint32_t sw_key(float x) {
  const uint32_t b = __float_as_uint(x);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
// a NaN logit counts as -inf; -0 and +0 are one value (their bit patterns differ)
__device__ __forceinline__ float sw_clean(float x) { return x != x ? -INFINITY : (x == 0.f ? 0.f : x); }

struct SwScale {
  float mx, inv_w, c, mc, z;               // row max, buckets per unit of x, log2(e)/T, mx*c, sum of e
};
// Every wave of every workgroup of a row computes this from the same numbers in the same order:
// lane c takes chunk c (S <= 64), and the lanes meet in a butterfly, which gives all of them
// the same bits.
__device__ __forceinline__ SwScale sw_scale(const SwRow& w, int S, float T, bool with_sum) {
  const int lane = threadIdx.x & 63;
  const float mx = wave_max(lane < S ? w.cmax[lane] : -INFINITY);
  const float mn = -wave_max(lane < S ? -w.cmin[lane] : -INFINITY);
  SwScale s;
  s.z = with_sum ? wave_sum(lane < S ? w.csum[lane] : 0.f) : 0.f;
  s.mx = mx;
  s.c = 1.4426950408889634f / T;
  s.mc = mx * s.c;
  const float span = fminf(mx - mn, SW_SPAN * T);
  s.inv_w = span > 0.f ? (float)SW_BUCKETS / span : 0.f;
  return s;
}
__device__ __forceinline__ float sw_exp(float x, const SwScale& s) {
  return __builtin_amdgcn_exp2f(fmaf(x, s.c, -s.mc));
}
__device__ __forceinline__ int sw_bucket(float x, const SwScale& s) {
  const float fb = (s.mx - x) * s.inv_w;                 // (NaN when -inf meets inv_w 0: bucket 0)
  return (int)fminf(fmaxf(fb, 0.f), (float)(SW_BUCKETS - 1));
}
__device__ __forceinline__ bool sw_kept(float x, const SwScale& s, int cross, uint32_t edge) {
  const int b = sw_bucket(x, s);
  return b < cross || (b == cross && sw_key(x) > edge);
}

// Parameters of the rows of a launch: in device memory, or by value from the host (a copy to the device would be a pinned
// allocation, a transfer and its place in the stream for 12 bytes a row).
#define SW_GROUP 64
struct SwParams {
  const float *temperature, *top_p, *uniform;      // null: by value
  float value[SW_GROUP][3];
};
__device__ __forceinline__ void sw_params(const SwParams& p, int r, int row0, float& t, float& top, float& u) {
  if (p.temperature) {
    t = p.temperature[row0 + r];
    top = p.top_p[row0 + r];
    u = p.uniform[row0 + r];
  } else {
    t = p.value[r][0];
    top = p.value[r][1];
    u = p.value[r][2];
  }
}

// The larger of two numbers each over the block; scratch holds 16 floats.
__device__ __forceinline__ void block_max2(float& a, float& b, float* scratch) {
  a = wave_max(a);
  b = wave_max(b);
  const int wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) { scratch[wave] = a; scratch[8 + wave] = b; }
  __syncthreads();
  a = scratch[0];
  b = scratch[8];
  for (int i = 1; i < nw; ++i) { a = fmaxf(a, scratch[i]); b = fmaxf(b, scratch[8 + i]); }
}

// A chunk's largest and smallest finite logit and, if ``candidates``, what the row's nucleus can be made of (a token left out
// has all of a mass above top_p before it). With e = exp(x/T - chunk max), z_c the chunk's sum, z the row's: tokens
// whose e is below (1 - top_p) z / V have together less than (1 - top_p) z, so the cumulative mass passes top_p above
// them; z_c is at most z in the same units, and half of that bound leaves room for rounding. Candidates go on in the
// order of the vocabulary: a thread has four consecutive tokens of each quarter of the chunk, and one scan counts all four quarters.
__global__ void __launch_bounds__(SW_THREADS)
sw_scan_kernel(float* __restrict__ ws, const float* __restrict__ logits, int V, long stride, int S, int row0, int candidates,
               const SwParams params) {
  constexpr int Q = SW_PER / 4;
  static_assert(Q == 4, "four counts of 16 bits");
  __shared__ float scratch[17];
  __shared__ unsigned long long counts[SW_THREADS / 64];
  const int r = blockIdx.y, c = blockIdx.x, tid = threadIdx.x;
  const SwRow w = sw_row(ws, row0 + r, S);
  float T, top_p, u;
  sw_params(params, r, row0, T, top_p, u);
  const float* row = logits + (size_t)(row0 + r) * stride;
  const int lo = c * SW_CHUNK;
  float x[Q][4];
  const bool whole = lo + SW_CHUNK <= V && (reinterpret_cast<uintptr_t>(row) & 15) == 0;
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int i = lo + 4 * (q * SW_THREADS + tid);
    if (whole) {
      const float4 v = *reinterpret_cast<const float4*>(row + i);
      x[q][0] = v.x; x[q][1] = v.y; x[q][2] = v.z; x[q][3] = v.w;
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) x[q][k] = i + k < V ? row[i + k] : -INFINITY;
    }
  }
  float mx = -INFINITY, neg = -INFINITY;
#pragma unroll
  for (int q = 0; q < Q; ++q)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      x[q][k] = sw_clean(x[q][k]);
      mx = fmaxf(mx, x[q][k]);
      if (x[q][k] > -INFINITY) neg = fmaxf(neg, -x[q][k]);
    }
  block_max2(mx, neg, scratch);
  if (tid == 0) {
    w.cmax[c] = mx;
    w.cmin[c] = -neg;
    if (c == 0) {
      w.result[7] = 0.f;
      w.result[8] = T;
      w.result[9] = top_p;
      w.result[10] = u;
    }
  }
  if (!candidates) return;
  if (!(top_p < 1.0f)) {                       // every token is kept: the other kernels
    if (tid == 0) w.ccount[c] = SW_SEG + 1;
    return;
  }
  // (as (x - max) c: with x c - (max c), one rounding of the product, a chunk's sum is off by 2^(2^-24 max c), 1 % where the largest
  // logit is 3e5 temperatures, and every chunk's by another factor)
  const float scale = 1.4426950408889634f / T;
  float e[Q][4], z = 0.f;
#pragma unroll
  for (int q = 0; q < Q; ++q)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      e[q][k] = mx > -INFINITY ? __builtin_amdgcn_exp2f((x[q][k] - mx) * scale) : 0.f;
      z += e[q][k];
    }
  z = block_sum(z, scratch);
  const float least = 0.5f * (1.0f - top_p) * z / (float)V;
  unsigned long long mine = 0ull;
#pragma unroll
  for (int q = 0; q < Q; ++q)
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (e[q][k] > 0.f && e[q][k] >= least) mine += 1ull << (16 * q);
  unsigned long long upto = mine;
  const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned long long n = __shfl_up(upto, o, 64);
    if (lane >= o) upto += n;
  }
  if (lane == 63) counts[wave] = upto;
  __syncthreads();
  unsigned long long before = upto - mine, all = 0ull;
#pragma unroll
  for (int i = 0; i < SW_THREADS / 64; ++i) {
    if (i < wave) before += counts[i];
    all += counts[i];
  }
  int first = 0;
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    int at = first + (int)((before >> (16 * q)) & 0xffff);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (e[q][k] > 0.f && e[q][k] >= least) {
        if (at < SW_SEG) {
          w.seg_x[(size_t)c * SW_SEG + at] = x[q][k];
          w.seg_i[(size_t)c * SW_SEG + at] = lo + 4 * (q * SW_THREADS + tid) + k;
        }
        ++at;
      }
    first += (int)((all >> (16 * q)) & 0xffff);
  }
  if (tid == 0) {
    w.csum[c] = z;
    w.ccount[c] = first;
  }
}

__global__ void __launch_bounds__(SW_THREADS)
sw_hist_kernel(float* __restrict__ ws, const float* __restrict__ logits, int V, long stride, int S) {
  __shared__ unsigned long long hist[SW_BUCKETS];
  __shared__ float scratch[16];
  const int r = blockIdx.y, c = blockIdx.x;
  const SwRow w = sw_row(ws, r, S);
  if (w.result[7] != 0.f) return;
  const float* row = logits + (size_t)r * stride;
  const SwScale s = sw_scale(w, S, w.result[8], false);
  for (int b = threadIdx.x; b < SW_BUCKETS; b += SW_THREADS) hist[b] = 0ull;
  __syncthreads();
  const int lo = c * SW_CHUNK;
  float x[SW_PER];
#pragma unroll
  for (int j = 0; j < SW_PER; ++j) {
    const int i = lo + j * SW_THREADS + threadIdx.x;
    x[j] = i < V ? sw_clean(row[i]) : -INFINITY;
  }
  float z = 0.f;
  unsigned long long last = 0ull;
#pragma unroll
  for (int j = 0; j < SW_PER; ++j) {
    const int i = lo + j * SW_THREADS + threadIdx.x;
    if (i < V) {
      const float e = sw_exp(x[j], s);
      z += e;
      const unsigned long long fixed = (unsigned long long)(e * SW_FIXED + 0.5f);
      const int b = sw_bucket(x[j], s);
      if (b == SW_BUCKETS - 1) last += fixed;
      else atomicAdd(&hist[b], fixed);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) last += __shfl_xor(last, o, 64);
  if ((threadIdx.x & 63) == 0) atomicAdd(&hist[SW_BUCKETS - 1], last);
  z = block_sum(z, scratch);               // (its barriers also complete the histogram)
  if (threadIdx.x == 0) w.csum[c] = z;
  float* out = w.hist + (size_t)c * SW_BUCKETS;
  for (int b = threadIdx.x; b < SW_BUCKETS; b += SW_THREADS) out[b] = (float)hist[b] * (1.0f / SW_FIXED);
}

// The bucket in which the mass, most likely tokens first, passes tp, and the mass before it;
// BUCKETS if it never does (everything is kept). The first SW_THREADS threads work, every
// thread of the block must call (barriers). tmp: 8 floats and 2 ints of LDS.
template <int BUCKETS>
__device__ __forceinline__ void sw_crossing(const float* tot, float tp, float* tmp, int* itmp, int* cross,
                                            float* before) {
  constexpr int PER = BUCKETS / SW_THREADS;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bool works = tid < SW_THREADS;
  float v[PER], mine = 0.f;
  if (works) {
#pragma unroll
    for (int j = 0; j < PER; ++j) { v[j] = tot[tid * PER + j]; mine += v[j]; }
  }
  float inc = mine;
  if (works) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float n = __shfl_up(inc, o, 64);
      if (lane >= o) inc += n;
    }
  }
  if (tid == 0) { itmp[0] = BUCKETS; }
  if (works && lane == 63) tmp[wave] = inc;
  __syncthreads();
  float run = 0.f;
  if (works) {
    for (int i = 0; i < wave; ++i) run += tmp[i];
    run += inc - mine;                     // mass before this thread's buckets
    int first = BUCKETS;
    float r2 = run;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      if (first == BUCKETS && r2 + v[j] > tp) first = tid * PER + j;
      if (first == BUCKETS) r2 += v[j];
    }
    if (first < BUCKETS) atomicMin(&itmp[0], first);
  }
  __syncthreads();
  const int cb = itmp[0];
  if (works && cb < BUCKETS && cb / PER == tid) {
    float r2 = run;
    for (int j = 0; j < cb - tid * PER; ++j) r2 += v[j];
    tmp[4] = r2;
  }
  __syncthreads();
  *cross = cb;
  *before = cb < BUCKETS ? tmp[4] : 0.f;
}

// One workgroup a row; a thread adds two buckets, eight chunks' loads under way, in chunk order.
#define SW_COMBINE_THREADS (SW_BUCKETS / 2)
__global__ void __launch_bounds__(SW_COMBINE_THREADS)
sw_combine_kernel(float* __restrict__ ws, int S) {
  __shared__ float tot[SW_BUCKETS];
  __shared__ float tmp[17];
  __shared__ int itmp[2];
  const int r = blockIdx.x;
  const SwRow w = sw_row(ws, r, S);
  if (w.result[7] != 0.f) return;
  const float top_p = w.result[9];
  const SwScale s = sw_scale(w, S, w.result[8], true);
  int cross = SW_BUCKETS;
  float before = 0.f;
  if (top_p < 1.0f) {
    float2 t = make_float2(0.f, 0.f);
    const float* mine = w.hist + 2 * threadIdx.x;
    for (int c0 = 0; c0 < S; c0 += 8) {
      float2 v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        // (rows of the workspace begin at any multiple of four bytes)
        const float* p = mine + (size_t)(c0 + j) * SW_BUCKETS;
        v[j] = c0 + j < S ? make_float2(p[0], p[1]) : make_float2(0.f, 0.f);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        t.x += v[j].x;
        t.y += v[j].y;
      }
    }
    tot[2 * threadIdx.x] = t.x;
    tot[2 * threadIdx.x + 1] = t.y;
    __syncthreads();
    sw_crossing<SW_BUCKETS>(tot, top_p * s.z, tmp, itmp, &cross, &before);
  }
  if (threadIdx.x == 0) {
    w.result[1] = __int_as_float(cross);
    w.result[3] = before;
    w.result[4] = s.mx;
    w.result[5] = s.inv_w;
    w.result[6] = s.z;
  }
}

// What the combine kernel found for a row.
__device__ __forceinline__ SwScale sw_found(const SwRow& w, float T, int* cross) {
  *cross = __float_as_int(w.result[1]);
  SwScale s;
  s.mx = w.result[4];
  s.inv_w = w.result[5];
  s.z = w.result[6];
  s.c = 1.4426950408889634f / T;
  s.mc = s.mx * s.c;
  return s;
}

__global__ void __launch_bounds__(SW_THREADS)
sw_gather_kernel(float* __restrict__ ws, const float* __restrict__ logits, int V, long stride, int S) {
  __shared__ float tmp[17];
  const int r = blockIdx.y, c = blockIdx.x;
  const SwRow w = sw_row(ws, r, S);
  if (w.result[7] != 0.f) return;
  const float* row = logits + (size_t)r * stride;
  int cross;
  const SwScale s = sw_found(w, w.result[8], &cross);
  const int lo = c * SW_CHUNK;
  float x[SW_PER];
#pragma unroll
  for (int j = 0; j < SW_PER; ++j) {
    const int i = lo + j * SW_THREADS + threadIdx.x;
    x[j] = i < V ? sw_clean(row[i]) : -INFINITY;
  }
  float sure = 0.f;
  int mine = 0;
  bool in[SW_PER];
#pragma unroll
  for (int j = 0; j < SW_PER; ++j) {
    const int i = lo + j * SW_THREADS + threadIdx.x;
    const int b = sw_bucket(x[j], s);
    in[j] = i < V && b == cross;
    if (i < V && b < cross) sure += sw_exp(x[j], s);
    mine += in[j] ? 1 : 0;
  }
  float total;
  const int at0 = (int)block_exclusive_scan((float)mine, tmp, &total);   // (counts up to 4096: exact)
  sure = block_sum(sure, tmp);
  if (threadIdx.x == 0) {
    w.ckept[c] = sure;
    w.ccount[c] = (int)total;
  }
  int at = at0;
#pragma unroll
  for (int j = 0; j < SW_PER; ++j) {
    if (in[j]) {
      if (at < SW_SEG) {
        w.seg_x[(size_t)c * SW_SEG + at] = x[j];
        w.seg_i[(size_t)c * SW_SEG + at] = lo + j * SW_THREADS + threadIdx.x;
      }
      ++at;
    }
  }
}

// inclusive prefix over the lanes of a wave, in a fixed order
__device__ __forceinline__ float wave_inclusive_scan(float v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float n = __shfl_up(v, o, 64);
    if (lane >= o) v += n;
  }
  return v;
}

// The edge of the nucleus among the n tokens of the crossing bucket, in LDS (kept: key > edge): the mass of all larger ones,
// added in list order, and what lies ``before`` the bucket is at most tp. A block of SW_THREADS; vote_key and vote_low: 4 words of LDS.
__device__ __forceinline__ uint32_t sw_edge(const float* list_x, const float* list_e, int n, float before, float tp,
                                            uint32_t* vote_key, int* vote_low) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t lo = 0u, hi = 0xffffffffu, edge;
  if (n <= SW_THREADS) {
    // Few tokens: every one of them asks directly whether it is kept (the mass of the
    // tokens above it, added in list order, and what lies before the bucket); the edge is
    // the smallest kept key, less one.
    uint32_t lowest = 0xffffffffu;
    for (int i = tid; i < n; i += SW_THREADS) {
      const uint32_t k = sw_key(list_x[i]);
      float mass = 0.f;
      for (int j = 0; j < n; ++j) mass += sw_key(list_x[j]) > k ? list_e[j] : 0.f;
      if (mass + before <= tp) lowest = min(lowest, k);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) lowest = min(lowest, (uint32_t)__shfl_xor((int)lowest, o, 64));
    if (lane == 0) vote_key[wave] = lowest;
    __syncthreads();
    lowest = min(min(vote_key[0], vote_key[1]), min(vote_key[2], vote_key[3]));
    edge = lowest - 1u;                // (no token kept: 0xfffffffe, nothing in the bucket passes)
    if (lowest == 0xffffffffu) edge = 0xffffffffu;
  } else {
    // The edge lies between the list's smallest key (less one: everything above it is the
    // whole list) and its largest (nothing above it). Four waves try four keys a round.
    uint32_t kmin = 0xffffffffu, kmax = 0u;
    for (int i = lane; i < n; i += 64) {
      const uint32_t k = sw_key(list_x[i]);
      kmin = min(kmin, k);
      kmax = max(kmax, k);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      kmin = min(kmin, (uint32_t)__shfl_xor((int)kmin, o, 64));
      kmax = max(kmax, (uint32_t)__shfl_xor((int)kmax, o, 64));
    }
    lo = kmin - 1u;
    hi = kmax;
    while (hi - lo > 1u) {
      // gap keys lie strictly between lo and hi; wave v tries one of them: all of them
      // when there are at most four, else four spread evenly
      const uint32_t gap = hi - lo - 1u;
      const bool mine = gap > 4u || (uint32_t)wave < gap;
      const uint32_t mid = gap > 4u
          ? lo + 1u + (uint32_t)(((unsigned long long)gap * (uint32_t)(wave + 1)) / 5u)
          : lo + 1u + (uint32_t)wave;
      float mass = 0.f;
      if (mine) {
        for (int i = lane; i < n; i += 64) mass += sw_key(list_x[i]) > mid ? list_e[i] : 0.f;
        mass = wave_sum(mass) + before;
      }
      __syncthreads();
      if (lane == 0) { vote_key[wave] = mine ? mid : 0u; vote_low[wave] = !mine ? -1 : (mass > tp ? 1 : 0); }
      __syncthreads();
      uint32_t nlo = lo, nhi = hi;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if (vote_low[v] == 1) nlo = max(nlo, vote_key[v]);
        if (vote_low[v] == 0) nhi = min(nhi, vote_key[v]);
      }
      lo = nlo; hi = nhi;
    }
    edge = lo;
  }
  return edge;
}

// The token of a row from its candidates alone, if there are few: what the kernels from hist to draw do, by one workgroup in
// LDS. Rows with more, or with more than SW_SMALL_LIST tokens in the crossing bucket, are left to those kernels, which leave at
// once from a row that is done.
#define SW_SMALL 4096
#define SW_SMALL_BUCKETS 1024
#define SW_SMALL_LIST 1024
__global__ void __launch_bounds__(SW_THREADS)
sw_small_kernel(int32_t* __restrict__ out, float* __restrict__ ws, int S) {
  __shared__ float tmp[17];
  __shared__ int itmp[2];
  __shared__ float cand[SW_SMALL];
  __shared__ int32_t token[SW_SMALL];
  __shared__ unsigned long long hist[SW_SMALL_BUCKETS];
  __shared__ float list_x[SW_SMALL_LIST], list_e[SW_SMALL_LIST];
  __shared__ int seg_at[65];
  __shared__ uint32_t vote_key[4];
  __shared__ int vote_low[4], choice_s, last_kept;
  float* const tot = list_x;               // (the buckets' sums are read before the list is made)
  static_assert(SW_SMALL_LIST >= SW_SMALL_BUCKETS, "one place for both");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = blockIdx.x;
  const SwRow w = sw_row(ws, r, S);
  const float T = w.result[8], top_p = w.result[9], u = w.result[10];
  const int count = lane < S ? w.ccount[lane] : 0;
  const float cmax = lane < S ? w.cmax[lane] : -INFINITY, csum = lane < S ? w.csum[lane] : 0.f;
  SwScale s = sw_scale(w, S, T, false);
  s.inv_w *= (float)SW_SMALL_BUCKETS / SW_BUCKETS;
  if (__any(count > SW_SEG) || !(s.mx > -INFINITY)) return;
  auto exp_of = [&](float x) { return __builtin_amdgcn_exp2f((x - s.mx) * s.c); };   // (as the chunks' sums have it)
  s.z = wave_sum(csum > 0.f ? csum * exp_of(cmax) : 0.f);
  const int upto = (int)wave_inclusive_scan((float)count);            // (small integers: exact)
  const int n = __shfl(upto, 63, 64);
  if (n > SW_SMALL) return;
  if (wave == 0 && lane < S) { seg_at[lane] = upto - count; seg_at[lane + 1] = upto; }
  for (int b = tid; b < SW_SMALL_BUCKETS; b += SW_THREADS) hist[b] = 0ull;
  if (tid == 0) { choice_s = -1; last_kept = -1; }
  __syncthreads();
  auto bucket = [&](float x) {
    return (int)fminf(fmaxf((s.mx - x) * s.inv_w, 0.f), (float)(SW_SMALL_BUCKETS - 1));
  };
  for (int c = tid >> 3; c < S; c += SW_THREADS / 8) {                // eight threads a chunk
    const int base = seg_at[c], k = seg_at[c + 1] - base;
    for (int j0 = tid & 7; j0 < k; j0 += 8 * 4) {                     // four loads of each under way
      float x[4];
      int32_t at[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = min(j0 + 8 * q, k - 1);
        x[q] = w.seg_x[(size_t)c * SW_SEG + j];
        at[q] = w.seg_i[(size_t)c * SW_SEG + j];
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = j0 + 8 * q;
        if (j >= k) continue;
        cand[base + j] = x[q];
        token[base + j] = at[q];
        atomicAdd(&hist[bucket(x[q])], (unsigned long long)(exp_of(x[q]) * SW_FIXED + 0.5f));
      }
    }
  }
  __syncthreads();
  for (int b = tid; b < SW_SMALL_BUCKETS; b += SW_THREADS) tot[b] = (float)hist[b] * (1.0f / SW_FIXED);
  __syncthreads();
  const float tp = top_p * s.z;
  int cross;
  float before;
  sw_crossing<SW_SMALL_BUCKETS>(tot, tp, tmp, itmp, &cross, &before);
  if (cross >= SW_SMALL_BUCKETS) return;   // (rounding, with top_p next to 1)
  // a thread has consecutive candidates from here on
  const int per = (n + SW_THREADS - 1) / SW_THREADS, a = min(n, per * tid), b = min(n, a + per);
  int mine = 0;
  for (int i = a; i < b; ++i) mine += bucket(cand[i]) == cross ? 1 : 0;
  float in_bucket;
  int at = (int)block_exclusive_scan((float)mine, tmp, &in_bucket);
  if (in_bucket > (float)SW_SMALL_LIST) return;
  for (int i = a; i < b; ++i)
    if (bucket(cand[i]) == cross) {
      list_x[at] = cand[i];
      list_e[at++] = exp_of(cand[i]);
    }
  __syncthreads();
  uint32_t edge = sw_edge(list_x, list_e, (int)in_bucket, before, tp, vote_key, vote_low);
  // the most likely token is always kept: nothing lies before it
  if (cross == 0 && edge >= sw_key(s.mx)) edge = sw_key(s.mx) - 1u;
  auto kept = [&](float x) {
    const int k = bucket(x);
    return k < cross || (k == cross && sw_key(x) > edge);
  };
  float mass = 0.f;
  int my_last = -1;
  for (int i = a; i < b; ++i)
    if (kept(cand[i])) {
      mass += exp_of(cand[i]);
      my_last = i;
    }
  float total;
  const float run = block_exclusive_scan(mass, tmp, &total);
  const float target = u * total;
  if (mass > 0.f && run <= target && target < run + mass) {
    int choice = my_last;
    float sum = run;
    for (int i = a; i < b; ++i)
      if (kept(cand[i])) {
        sum += exp_of(cand[i]);
        if (sum > target) { choice = i; break; }
      }
    choice_s = choice;
  }
  if (my_last >= 0) atomicMax(&last_kept, my_last);
  __syncthreads();
  // rounding may leave the target past the last kept token: take that token
  if (tid == 0) {
    out[r] = token[choice_s >= 0 ? choice_s : last_kept];
    w.result[7] = 1.f;
  }
}

__global__ void __launch_bounds__(SW_THREADS)
sw_draw_kernel(int32_t* __restrict__ out, float* __restrict__ ws, const float* __restrict__ logits, int V,
               long stride, int S) {
  __shared__ float tmp[17];
  __shared__ float list_x[SW_LIST], list_e[SW_LIST];
  __shared__ int seg_at[65];
  __shared__ uint32_t edge_s, vote_key[4];
  __shared__ int vote_low[4];
  __shared__ int pick_chunk, last_kept, choice_s;
  __shared__ float pick_before, kept_s;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = blockIdx.x;
  const SwRow w = sw_row(ws, r, S);
  const float* row = logits + (size_t)r * stride;
  int cross;
  if (w.result[7] != 0.f) return;
  const SwScale s = sw_found(w, w.result[8], &cross);
  const float before = w.result[3];
  const float tp = w.result[9] * s.z, uniform = w.result[10];
  const int my_count = lane < S ? w.ccount[lane] : 0;
  const float my_sure = lane < S ? w.ckept[lane] : 0.f;
  if (tid == 0) { last_kept = -1; choice_s = -1; }

  uint32_t edge = 0u;                      // kept inside the crossing bucket: key > edge
  bool whole_row = false;
  int n = 0;
  if (cross < SW_BUCKETS) {
    // where every chunk's tokens go in the list (every wave computes the same)
    const int fits = min(my_count, SW_SEG);
    const int upto = (int)wave_inclusive_scan((float)fits);          // (small integers: exact)
    n = __shfl(upto, 63, 64);
    whole_row = __any(my_count > SW_SEG) || n > SW_LIST;
    if (wave == 0 && lane < S) { seg_at[lane] = upto - fits; seg_at[lane + 1] = upto; }
    __syncthreads();
    // lo keeps mass_above(lo) > tp, hi keeps mass_above(hi) <= tp (mass_above counts key > t)
    uint32_t lo = 0u, hi = 0xffffffffu;
    if (!whole_row) {
      for (int c = tid >> 3; c < S; c += SW_THREADS / 8) {            // eight threads a chunk
        const int base = seg_at[c], k = seg_at[c + 1] - base;
        for (int j = tid & 7; j < k; j += 8) {
          const float x = w.seg_x[(size_t)c * SW_SEG + j];
          list_x[base + j] = x;
          list_e[base + j] = sw_exp(x, s);
        }
      }
      __syncthreads();
      edge = sw_edge(list_x, list_e, n, before, tp, vote_key, vote_low);
    } else {                               // too many tokens in one bucket: bisect over the whole row
      while (hi - lo > 1u) {
        const uint32_t mid = lo + ((hi - lo) >> 1);
        float mass = 0.f;
        for (int i = tid; i < V; i += SW_THREADS) {
          const float x = sw_clean(row[i]);
          if (sw_bucket(x, s) == cross && sw_key(x) > mid) mass += sw_exp(x, s);
        }
        mass = block_sum(mass, tmp) + before;
        if (mass <= tp) hi = mid; else lo = mid;
      }
      edge = lo;
    }
    // the most likely token is always kept: nothing lies before it
    if (cross == 0 && edge >= sw_key(s.mx)) edge = sw_key(s.mx) - 1u;
  }

  // kept mass chunk by chunk: what lies above the crossing bucket, and the kept part of it;
  // wave 0 (lane c: chunk c) adds them up and finds the chunk that holds the target
  float extra = 0.f;
  if (whole_row) {
    for (int c = 0; c < S; ++c) {
      float part = 0.f;
      for (int i = c * SW_CHUNK + tid; i < min(V, (c + 1) * SW_CHUNK); i += SW_THREADS) {
        const float x = sw_clean(row[i]);
        if (sw_bucket(x, s) == cross && sw_key(x) > edge) part += sw_exp(x, s);
      }
      part = block_sum(part, tmp);
      if (lane == c) extra = part;
    }
  } else if (cross < SW_BUCKETS && lane < S) {
    for (int j = seg_at[lane]; j < seg_at[lane + 1]; ++j) extra += sw_key(list_x[j]) > edge ? list_e[j] : 0.f;
  }
  if (wave == 0) {
    const float mass = my_sure + extra;
    const float upto = wave_inclusive_scan(mass);
    const float kept = __shfl(upto, 63, 64);
    const float target = uniform * kept;
    const unsigned long long holds = __ballot(mass > 0.f && upto > target);
    const unsigned long long any = __ballot(mass > 0.f);
    if (lane == 0) {
      int pc;
      if (holds) {
        pc = __ffsll((long long)holds) - 1;
      } else {                             // rounding: past the last kept token
        pc = any ? 63 - __clzll((long long)any) : 0;
      }
      pick_chunk = pc;
      kept_s = kept;
      w.result[0] = __uint_as_float(edge);
      w.result[2] = kept;
    }
    if (holds && lane == __ffsll((long long)holds) - 1) pick_before = upto - mass;
    if (!holds && lane == 0) pick_before = -INFINITY;
  }
  __syncthreads();
  // walk the chunk that holds the target: sixteen consecutive tokens a thread
  const int c0 = pick_chunk * SW_CHUNK;
  const float target = uniform * kept_s - pick_before;
  float xv[SW_PER], v[SW_PER], mine = 0.f;
  int my_last = -1;
#pragma unroll
  for (int k = 0; k < SW_PER; ++k) {
    const int i = c0 + SW_PER * tid + k;
    xv[k] = i < V ? sw_clean(row[i]) : -INFINITY;
    v[k] = i < V ? sw_exp(xv[k], s) : 0.f;
  }
#pragma unroll
  for (int k = 0; k < SW_PER; ++k) {
    const int i = c0 + SW_PER * tid + k;
    // (as a select: written as "if (!(...)) v[k] = 0" this loop kept what it should drop)
    const bool keep = i < V && sw_kept(xv[k], s, cross, edge);
    v[k] = keep ? v[k] : 0.f;
    if (v[k] > 0.f) my_last = i;
    mine += v[k];
  }
  float total;
  const float run = block_exclusive_scan(mine, tmp, &total);
  if (mine > 0.f && run <= target && target < run + mine) {
    int choice = my_last;
    float upto = run;
    bool found = false;
#pragma unroll
    for (int k = 0; k < SW_PER; ++k) {
      upto += v[k];
      if (!found && v[k] > 0.f && upto > target) { choice = c0 + SW_PER * tid + k; found = true; }
    }
    choice_s = choice;
  }
  if (my_last >= 0) atomicMax(&last_kept, my_last);
  __syncthreads();
  // rounding may leave the target past the chunk's last kept token: take that token
  if (tid == 0) out[r] = choice_s >= 0 ? choice_s : max(last_kept, 0);
}

__global__ void __launch_bounds__(SW_THREADS)
sw_probs_kernel(float* __restrict__ ws, float* __restrict__ work, const float* __restrict__ logits,
                int V, long stride, int S) {
  const int r = blockIdx.y, c = blockIdx.x;
  const SwRow w = sw_row(ws, r, S);
  const float* row = logits + (size_t)r * stride;
  float* ex = work + (size_t)r * V;
  int cross;
  const SwScale s = sw_found(w, w.result[8], &cross);
  const uint32_t edge = __float_as_uint(w.result[0]);
  const float inv_kept = 1.0f / w.result[2];
#pragma unroll
  for (int j = 0; j < SW_PER; ++j) {
    const int i = c * SW_CHUNK + j * SW_THREADS + threadIdx.x;
    if (i >= V) continue;
    const float x = sw_clean(row[i]);
    ex[i] = sw_kept(x, s, cross, edge) ? sw_exp(x, s) * inv_kept : 0.f;
  }
}

// bytes of workspace ptl_sample_top_p_wide needs for R rows of V logits
extern "C" size_t ptl_sample_top_p_wide_workspace(int R, int V) {
  const int S = (V + SW_CHUNK - 1) / SW_CHUNK;
  return (size_t)R * sw_row_words(S) * sizeof(float);
}

static int sample_wide(int32_t* out, float* work, int want_probs, const float* logits, int R, int V, long stride,
                       const SwParams& params, const float* values, float* ws, hipStream_t stream) {
  const int S = (V + SW_CHUNK - 1) / SW_CHUNK;
  const dim3 chunks(S, R);
  for (int row0 = 0; row0 < R; row0 += SW_GROUP) {
    const int rows = R - row0 < SW_GROUP ? R - row0 : SW_GROUP;
    SwParams p = params;
    if (values) memcpy(p.value, values + (size_t)3 * row0, (size_t)rows * 3 * sizeof(float));
    sw_scan_kernel<<<dim3(S, rows), SW_THREADS, 0, stream>>>(ws, logits, V, stride, S, row0, !want_probs, p);
  }
  // (with the probabilities of all tokens the nucleus is wanted in the form that the last kernel reads)
  if (!want_probs) sw_small_kernel<<<R, SW_THREADS, 0, stream>>>(out, ws, S);
  sw_hist_kernel<<<chunks, SW_THREADS, 0, stream>>>(ws, logits, V, stride, S);
  sw_combine_kernel<<<R, SW_COMBINE_THREADS, 0, stream>>>(ws, S);
  sw_gather_kernel<<<chunks, SW_THREADS, 0, stream>>>(ws, logits, V, stride, S);
  sw_draw_kernel<<<R, SW_THREADS, 0, stream>>>(out, ws, logits, V, stride, S);
  if (want_probs) sw_probs_kernel<<<chunks, SW_THREADS, 0, stream>>>(ws, work, logits, V, stride, S);
  return ptl_launch_status();
}

// As ptl_sample_top_p (work: only for the probabilities, if wanted); ws:
// ptl_sample_top_p_wide_workspace(R, V) bytes, 16-byte aligned.
// Rows of up to 64 chunks (262,144 logits).
extern "C" int ptl_sample_top_p_wide(int32_t* out, float* work, int want_probs, const float* logits,
                                     int R, int V, long stride, const float* temperature,
                                     const float* top_p, const float* uniform, float* ws,
                                     hipStream_t stream) {
  if (R <= 0) return PTL_OK;
  const int S = (V + SW_CHUNK - 1) / SW_CHUNK;
  if (V <= 0 || stride < V || (want_probs && !work) || !ws || S > 64 || R > 65535 || !temperature || !top_p || !uniform)
    return PTL_ERR_ARG;
  SwParams params{};
  params.temperature = temperature;
  params.top_p = top_p;
  params.uniform = uniform;
  return sample_wide(out, work, want_probs, logits, R, V, stride, params, nullptr, ws, stream);
}

// BLAKE2b (RFC 7693) without a key, the first 8 bytes of a digest of that length as a little-endian number.
static uint64_t blake2b_8(const uint8_t* text, size_t length) {
  static const uint64_t iv[8] = {0x6a09e667f3bcc908ull, 0xbb67ae8584caa73bull, 0x3c6ef372fe94f82bull, 0xa54ff53a5f1d36f1ull,
                                 0x510e527fade682d1ull, 0x9b05688c2b3e6c1full, 0x1f83d9abfb41bd6bull, 0x5be0cd19137e2179ull};
  static constexpr uint8_t sigma[10][16] = {
      {0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15}, {14, 10, 4, 8, 9, 15, 13, 6, 1, 12, 0, 2, 11, 7, 5, 3},
      {11, 8, 12, 0, 5, 2, 15, 13, 10, 14, 3, 6, 7, 1, 9, 4}, {7, 9, 3, 1, 13, 12, 11, 14, 2, 6, 5, 10, 4, 0, 15, 8},
      {9, 0, 5, 7, 2, 4, 10, 15, 14, 1, 11, 12, 6, 8, 3, 13}, {2, 12, 6, 10, 0, 11, 8, 3, 4, 13, 7, 5, 15, 14, 1, 9},
      {12, 5, 1, 15, 14, 13, 4, 10, 0, 7, 6, 3, 9, 2, 8, 11}, {13, 11, 7, 14, 12, 1, 3, 9, 5, 0, 15, 4, 8, 6, 2, 10},
      {6, 15, 14, 9, 11, 3, 0, 8, 12, 2, 13, 7, 1, 4, 10, 5}, {10, 2, 8, 4, 7, 6, 1, 5, 15, 11, 9, 14, 3, 12, 13, 0}};
  uint64_t h[8];
  memcpy(h, iv, sizeof(h));
  h[0] ^= 0x01010000ull ^ 8ull;
  size_t done = 0;
  do {
    const size_t n = length - done < 128 ? length - done : 128;
    uint64_t m[16] = {};
    memcpy(m, text + done, n);                   // (this host is little-endian too)
    done += n;
    uint64_t v[16];
    memcpy(v, h, sizeof(h));
    memcpy(v + 8, iv, sizeof(iv));
    v[12] ^= done;
    if (done == length) v[14] = ~v[14];
    auto mix = [&](int a, int b, int c, int d, uint64_t x, uint64_t y) {
      auto turn = [](uint64_t w, int k) { return (w >> k) | (w << (64 - k)); };
      v[a] += v[b] + x;
      v[d] = turn(v[d] ^ v[a], 32);
      v[c] += v[d];
      v[b] = turn(v[b] ^ v[c], 24);
      v[a] += v[b] + y;
      v[d] = turn(v[d] ^ v[a], 16);
      v[c] += v[d];
      v[b] = turn(v[b] ^ v[c], 63);
    };
#pragma unroll                                   // (the places of the words are known then: half the time)
    for (int round = 0; round < 12; ++round) {
      const uint8_t* at = sigma[round % 10];
#pragma unroll
      for (int i = 0; i < 4; ++i) mix(i, 4 + i, 8 + i, 12 + i, m[at[2 * i]], m[at[2 * i + 1]]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        mix(i, 4 + (i + 1) % 4, 8 + (i + 2) % 4, 12 + (i + 3) % 4, m[at[8 + 2 * i]], m[at[9 + 2 * i]]);
    }
    for (int i = 0; i < 8; ++i) h[i] ^= v[i] ^ v[8 + i];
  } while (done < length);
  return h[0];
}

// values[i][2] = a number in [0, 1) that depends on text i alone (texts one after the other, ends[i]: where the i-th ends)
extern "C" int ptl_uniforms(float* values, const uint8_t* texts, const int32_t* ends, int n) {
  int at = 0;
  for (int i = 0; i < n; ++i) {
    if (ends[i] < at) return PTL_ERR_ARG;
    values[3 * (size_t)i + 2] = (float)((double)(blake2b_8(texts + at, (size_t)(ends[i] - at)) >> 11) * (1.0 / 9007199254740992.0));
    at = ends[i];
  }
  return PTL_OK;
}

// The same without probabilities, temperature and top_p of every row in host memory ([R][3], the third made here of the row's
// text: ptl_uniforms); they are in the launch when the call returns.
extern "C" int ptl_sample_top_p_rows(int32_t* out, const float* logits, int R, int V, long stride, float* values,
                                     const uint8_t* texts, const int32_t* ends, float* ws, hipStream_t stream) {
  if (R <= 0) return PTL_OK;
  const int S = (V + SW_CHUNK - 1) / SW_CHUNK;
  if (V <= 0 || stride < V || !ws || S > 64 || R > 65535 || !values || !texts || !ends) return PTL_ERR_ARG;
  if (ptl_uniforms(values, texts, ends, R) != PTL_OK) return PTL_ERR_ARG;
  return sample_wide(out, nullptr, 0, logits, R, V, stride, SwParams{}, values, ws, stream);
}

// ptl_token_logprob: out[r] = log_softmax(logits[r])[tokens[r]], the log-probability the
// reference reports for a generated token (F.log_softmax of the step's logits gathered at
// the token, lite_llama/generete_with_probs.py:154-165). Rows of up to LP_ONE logits: one workgroup a row with the
// row in registers, one launch, no workspace. Longer ones: a workgroup a chunk of a row finds the chunk's max and its
// sum of exp(x - max); a wave a row puts the chunks together. (A workgroup reads a row of 128k logits at a small
// part of what the chip delivers: 64 rows 78 us, by chunks 10. At 32,000 logits the chunks take 5.7 to 6.5 us on
// the device and this form 7.1 to 7.5, but the second launch and the workspace cost the host 4 us, and a greedy
// pass with log-probabilities is bound by the host there: 26.3 us by chunks, 22.6 so; one MI355X.)
#define LP_ONE 32768
__global__ void __launch_bounds__(1024)
token_logprob_one_kernel(float* __restrict__ out, const float* __restrict__ logits, const int32_t* __restrict__ tokens,
                         int V, long stride) {
  constexpr int PER = LP_ONE / 1024;
  __shared__ float scratch[16];
  const float* row = logits + (size_t)blockIdx.x * stride;
  float x[PER], mx = -INFINITY;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = j * 1024 + threadIdx.x;
    x[j] = i < V ? row[i] : -INFINITY;
    mx = fmaxf(mx, x[j]);
  }
  mx = block_max(mx, scratch);
  float z = 0.f;
#pragma unroll
  for (int j = 0; j < PER; ++j) z += expf(x[j] - mx);
  z = block_sum(z, scratch);
  if (threadIdx.x == 0) {
    const int t = tokens[blockIdx.x];
    out[blockIdx.x] = (t >= 0 && t < V) ? row[t] - mx - logf(z) : -INFINITY;
  }
}

#define LP_CHUNK 4096
#define LP_THREADS 256
__global__ void __launch_bounds__(LP_THREADS)
token_logprob_part_kernel(float2* __restrict__ parts, int chunks, const float* __restrict__ logits, int V, long stride) {
  constexpr int PER = LP_CHUNK / LP_THREADS;
  __shared__ float scratch[16];
  const float* row = logits + (size_t)blockIdx.x * stride;
  for (int c = blockIdx.y; c < chunks; c += gridDim.y) {
    float x[PER], mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int i = c * LP_CHUNK + j * LP_THREADS + threadIdx.x;
      x[j] = i < V ? row[i] : -INFINITY;
      mx = fmaxf(mx, x[j]);
    }
    mx = block_max(mx, scratch);
    const float at = mx == -INFINITY ? 0.f : mx;     // (a chunk of -inf adds nothing)
    float z = 0.f;
#pragma unroll
    for (int j = 0; j < PER; ++j) z += expf(x[j] - at);
    z = block_sum(z, scratch);
    if (threadIdx.x == 0) parts[(size_t)blockIdx.x * chunks + c] = make_float2(mx, z);
  }
}

__global__ void __launch_bounds__(64)
token_logprob_kernel(float* __restrict__ out, const float2* __restrict__ parts, int chunks,
                     const float* __restrict__ logits, const int32_t* __restrict__ tokens, int V, long stride) {
  const int r = blockIdx.x, lane = threadIdx.x;
  parts += (size_t)r * chunks;
  float mx = -INFINITY, z = 0.f;
  for (int c = lane; c < chunks; c += 64) mx = fmaxf(mx, parts[c].x);
  mx = wave_max(mx);
  for (int c = lane; c < chunks; c += 64) z += parts[c].y * expf(parts[c].x - mx);
  z = wave_sum(z);
  if (lane == 0) {
    const int t = tokens[r];
    out[r] = (t >= 0 && t < V) ? logits[(size_t)r * stride + t] - mx - logf(z) : -INFINITY;
  }
}

// parts: of rows of more than 32,768 logits ceil(V / 4096) * 2 floats a row, 8-byte aligned
extern "C" int ptl_token_logprob(float* out, float* parts, const float* logits, const int32_t* tokens, int R, int V,
                                 long stride, hipStream_t stream) {
  if (R <= 0) return PTL_OK;
  if (V <= 0 || V > 0x7fffffff - LP_CHUNK || stride < V || (V > LP_ONE && !parts)) return PTL_ERR_ARG;
  if (V <= LP_ONE) {
    token_logprob_one_kernel<<<R, 1024, 0, stream>>>(out, logits, tokens, V, stride);
    return ptl_launch_status();
  }
  const int chunks = (V + LP_CHUNK - 1) / LP_CHUNK;
  token_logprob_part_kernel<<<dim3(R, chunks < 65535 ? chunks : 65535), LP_THREADS, 0, stream>>>(
      (float2*)parts, chunks, logits, V, stride);
  token_logprob_kernel<<<R, 64, 0, stream>>>(out, (const float2*)parts, chunks, logits, tokens, V, stride);
  return ptl_launch_status();
}
