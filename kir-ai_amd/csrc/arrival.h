// Partial results that the last workgroup to arrive combines in the launch that made them.
//
// The partials cross XCDs, whose L2s are not coherent with each other, so they are stored and
// loaded at agent scope (written through, and read past, the L2).  A wavefront waits until its
// stores have completed before its workgroup counts itself in, so whoever counts the last
// arrival finds every partial in memory; no release or acquire fence is needed beyond that (a
// release at agent scope writes the whole L2 back, ~0.45 us each, one after the other on an
// XCD).  The last workgroup sets the counter back for the next launch.
#pragma once

#include "wave_ops.h"

namespace llh {

__device__ __forceinline__ void st_agent(float *p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(float2 *p, float2 v) {
  __hip_atomic_store(reinterpret_cast<uint64_t *>(p), __builtin_bit_cast(uint64_t, v), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float ld_agent(const float *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float2 ld_agent(const float2 *p) {
  return __builtin_bit_cast(float2, __hip_atomic_load(reinterpret_cast<const uint64_t *>(p), __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT));
}

// Whether the calling workgroup is the last of n to count itself in (all its threads call).
__device__ __forceinline__ bool last_to_arrive(int32_t *counter, int n) {
  __shared__ int s_last;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's partials have reached memory
  __syncthreads();
  if (threadIdx.x == 0) {
    const int seen = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = seen == n - 1;
    if (seen == n - 1) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  return s_last != 0;
}

// U row parts of 128 dims, two a lane, each merged from its n <= 64 partials at agent scope:
// partial i of part u has its (max, sum) at ml[u] + i * ml_stride and its dims at
// o[u] + i * o_stride.  mx[u], sum[u]: the merged (max, sum), out[u]: this lane's dims.
// STEP partials of every part are in flight together.
template <int U, int STEP>
__device__ __forceinline__ void merge_parts(const float2 *const (&ml)[U], size_t ml_stride, const float *const (&o)[U],
                                            size_t o_stride, int n, int lane, float2 (&out)[U], float (&mx)[U],
                                            float (&sum)[U]) {
  static_assert(64 % STEP == 0, "the weights of a step lie in one wavefront");
  float2 pair[U], v[U][STEP];
  float f[U][1];
#pragma unroll
  for (int u = 0; u < U; u++) pair[u] = ld_agent(ml[u] + min(lane, n - 1) * ml_stride);
  for (int i0 = 0; i0 < n; i0 += STEP) {
#pragma unroll
    for (int i = 0; i < STEP; i++)
      if (i0 + i < n) {
#pragma unroll
        for (int u = 0; u < U; u++)
          v[u][i] = ld_agent(reinterpret_cast<const float2 *>(o[u] + (i0 + i) * o_stride) + lane);
      }
    if (i0 == 0) {
#pragma unroll
      for (int u = 0; u < U; u++) {
        const float m[1] = {lane < n ? pair[u].x : -INFINITY}, l[1] = {pair[u].y};
        sum[u] = merge_weights<1>(m, l, lane, f[u], &mx[u]);
        out[u] = make_float2(0.0f, 0.0f);
      }
    }
#pragma unroll
    for (int i = 0; i < STEP; i++)
      if (i0 + i < n) {
#pragma unroll
        for (int u = 0; u < U; u++) {
          const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f[u][0]), i0 + i));
          out[u].x += v[u][i].x * w;
          out[u].y += v[u][i].y * w;
        }
      }
  }
}

}  // namespace llh
