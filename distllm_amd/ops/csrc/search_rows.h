// Numbers in float32's order, and products of a query with rows of a corpus (search
// kernels).
#pragma once
#include "common.h"

__device__ __forceinline__ unsigned int f32_to_ord(float f) {
  union { float f; unsigned int u; } c;
  c.f = f;
  return (c.u & 0x80000000u) ? ~c.u : (c.u | 0x80000000u);
}
__device__ __forceinline__ float ord_to_f32(unsigned int u) {
  union { float f; unsigned int u; } c;
  c.u = (u & 0x80000000u) ? (u & 0x7fffffffu) : ~u;
  return c.f;
}

// Products of a query with rows r0 to r0 + 3 of a corpus by one wave: a lane sums
// every 64th four of columns, the lanes pairwise. Rows past the last are its.
__device__ __forceinline__ void search_dot(const float* query,
                                           const float* corpus, int r0, int N,
                                           int K, float (&s)[4]) {
  const float* from[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    from[r] = corpus + (long)min(r0 + r, N - 1) * K;
    s[r] = 0.f;
  }
#pragma unroll 3
  for (int c = (threadIdx.x & 63) * 4; c < K; c += 256) {
    const f32x4 y = *reinterpret_cast<const f32x4*>(query + c);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(from[r] + c);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[r] = fmaf(x[e], y[e], s[r]);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) s[r] = wave_reduce_sum(s[r]);
}
