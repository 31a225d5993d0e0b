// Residual sum and RMS norm of one row ahead of a product of it, in every
// workgroup of the product: h = (a + b) / rms(a + b) * w as bf16 numbers in
// LDS, a + b to memory from the first workgroup. A launch of its own for the
// norm is 3 us in which no weights come; here the rows' 16 KiB come from L2
// while the first weights are on their way. Sums and roundings are those of
// norm_fwd_small_kernel, bit for bit.
#pragma once
#include "common.h"

struct NormRow {
  const unsigned short *a, *b, *w;
  unsigned short* sum;
  float eps;
};

// 256 threads, K <= 2048 NC numbers, K % 8 == 0. red: 4 floats of LDS. start()
// issues the first copies of the weights: straight-line code, so that the
// compiler can count them and waits only for the loads ahead of them.
template <int NC, typename F>
__device__ __forceinline__ void norm_row(const NormRow& n, int K, float* red,
                                         char* hs, const F& start) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  s16x8 av[NC], bv[NC], wv[NC];
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const int c = min((int)(threadIdx.x + k * 256) * 8, K - 8);
    av[k] = *reinterpret_cast<const s16x8*>(n.a + c);
    bv[k] = *reinterpret_cast<const s16x8*>(n.b + c);
    wv[k] = *reinterpret_cast<const s16x8*>(n.w + c);
  }
  __builtin_amdgcn_sched_barrier(0);
  start();
  __builtin_amdgcn_sched_barrier(0);
  float x[NC][8], sumsq = 0.f;
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const int c = (threadIdx.x + k * 256) * 8;
    float t[8];
    bf8_to_f32(av[k], x[k]);
    bf8_to_f32(bv[k], t);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      x[k][i] += t[i];
      if (c < K) sumsq += x[k][i] * x[k][i];
    }
  }
  sumsq = wave_reduce_sum(sumsq);
  if (lane == 0) red[wid] = sumsq;
  // only LDS is waited for: the copies go on
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  const float inv =
      rsqrtf((red[0] + red[1] + red[2] + red[3]) / K + n.eps);
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const int c = (threadIdx.x + k * 256) * 8;
    if (c < K) {
      float wf[8];
      bf8_to_f32(wv[k], wf);
      s16x8 o, sv;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        o[i] = (short)f2bf(x[k][i] * inv * wf[i]);
        sv[i] = (short)f2bf(x[k][i]);
      }
      *reinterpret_cast<s16x8*>(hs + c * 2) = o;
      if (blockIdx.x == 0) *reinterpret_cast<s16x8*>(n.sum + c) = sv;
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
