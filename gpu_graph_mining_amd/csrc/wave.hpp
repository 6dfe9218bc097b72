// wave.hpp -- device helpers of the level-step kernels: one workgroup is one
// 64-lane wave, so a barrier is a compiler fence and scans are shuffles.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.hpp"

namespace gm {

constexpr int kSupShift = 40;  // packed counters: support << 40 | embeddings

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <class T>
__device__ __forceinline__ T wave_exclusive_scan(T x, T &total) {
  const int lane = threadIdx.x & 63;
  T v = x;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const T y = __shfl_up(v, o, 64);
    if (lane >= o) v += y;
  }
  total = __shfl(v, 63, 64);
  return v - x;
}

template <class T>
__device__ __forceinline__ T wave_sum(T x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}

__device__ __forceinline__ int wave_max(int x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x = max(x, __shfl_xor(x, o, 64));
  return x;
}

__device__ __forceinline__ uint64_t lanes_below(int lane) { return (1ull << lane) - 1ull; }

// Wall-clock stamps of the extension + support stage: the first chunks
// record ~start (the max of complements is the earliest start), every
// chunk its end; the host reads them from the spread lines.
__device__ __forceinline__ void stamp_start(unsigned long long *spread, int64_t ci) {
  if (ci < kSpread && threadIdx.x == 0)
    atomicMax(&spread[ci * kSpreadStride + kSpreadStart], ~(unsigned long long)__builtin_amdgcn_s_memrealtime());
}
__device__ __forceinline__ void stamp_end(unsigned long long *spread, int64_t ci) {
  if (threadIdx.x == 0)
    atomicMax(&spread[(ci & (kSpread - 1)) * kSpreadStride + kSpreadEnd],
              (unsigned long long)__builtin_amdgcn_s_memrealtime());
}

// Lane t's segment head within the block: the last segment start at or
// before t (0 when the segment began in an earlier block).
__device__ __forceinline__ int head_lane(uint64_t starts, int lane) {
  const uint64_t upto = starts & (lane == 63 ? ~0ull : ((2ull << lane) - 1ull));
  return upto ? 63 - __clzll((long long)upto) : 0;
}

// The level's counters start from zero: frequent-key count, failure list,
// errors and spread statistics but the written-row slots, which keep
// counting across levels (the host compares their total with the rows it
// asked for).
__device__ __forceinline__ void clear_counters(const StepArgs &a) {
  if (threadIdx.x == 0) {
    *a.freq_count = 0;
    *a.fail_count = 0;
    *a.error_flag = 0;
  }
  for (int i = threadIdx.x; i < kSpread * kSpreadStride; i += blockDim.x)
    if (i % kSpreadStride != kSpreadWritten) a.spread[i] = 0;
}

}  // namespace gm
