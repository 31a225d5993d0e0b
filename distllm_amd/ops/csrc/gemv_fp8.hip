// W8A16 projection GEMV for the interactive-decode regime:
//   out[M, N] = x[M, K] (bf16) @ (W_q[N, K] (fp8 e4m3) * scale[N])^T
// with optional bf16 bias. M <= 8 (per-token decode batches).
//
// The M=1 decode step is weight-stream bound (profiles/RESULTS.md "B=1
// interactive decode"): fp8 weights halve the HBM bytes per step. Scales are
// per output channel and applied after the fp32 dot: dot(w_q*s, x) == s *
// dot(w_q, x), so quantization only rounds the weights, never the
// accumulation.
//
// The ring kernel takes K % 128 == 0: a workgroup has 16 columns (of a gated
// unit 16 gate and the 16 up columns), its 4 waves take the 128-wide chunks of
// K in turn, W (2 KiB a chunk) and x (4 or 8 rows) pass through LDS buffers of
// the wave's own by global_load_lds, three or four chunks ahead, and W is widened
// to bf16 (exact) on its way to the MFMA. The vector-unit kernel above it, a
// wave per column with one 16-byte load a lane in flight, keeps the other K and
// one row of few columns. Measured in a decode graph, us: 28672 x 4096 with
// swiglu 31 + 5 -> 24.6, 4096 x 14336 and 4096 x 4096 together 29 -> 19, 6144 x
// 4096 9.8 -> 7.6.
// Reference anchor: the vLLM latency role the reference delegated
// (distllm/generate/generators/vllm_backend.py:62-93).
#include <hip/hip_fp8.h>

#include "norm_row.h"

#define GV_MAXM 8

__device__ __forceinline__ float gv_fp8(unsigned char u) {
  __hip_fp8_e4m3 v;
  v.__x = u;
  return float(v);
}

__global__ void __launch_bounds__(512)
gemv_fp8_kernel(const unsigned short* __restrict__ X,
                const unsigned char* __restrict__ W,
                const float* __restrict__ scale,
                const unsigned short* __restrict__ bias,
                unsigned short* __restrict__ OUT, int M, int N, long K) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = threadIdx.x >> 6;
  const int n = blockIdx.x * 8 + wid;  // one wave per output column
  if (n >= N) return;
  const unsigned char* w = W + (long)n * K;
  float acc[GV_MAXM];
#pragma unroll
  for (int m = 0; m < GV_MAXM; ++m) acc[m] = 0.f;

  const int niter = (int)((K + 1023) >> 10);  // K % 16 enforced host-side
  for (int it = 0; it < niter; ++it) {
    const long off = (long)it * 1024 + lane * 16;  // fp8-element offset
    if (off >= K) break;  // tail chunk: inactive lanes
    const uint4 wb = *reinterpret_cast<const uint4*>(w + off);
    const unsigned char* wp =
        reinterpret_cast<const unsigned char*>(&wb);
    float wf[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) wf[i] = gv_fp8(wp[i]);
    for (int m = 0; m < M; ++m) {
      const unsigned short* xr = X + (long)m * K + off;
      const uint4 xa = *reinterpret_cast<const uint4*>(xr);
      const uint4 xb = *reinterpret_cast<const uint4*>(xr + 8);
      const unsigned short* xp =
          reinterpret_cast<const unsigned short*>(&xa);
      const unsigned short* xq =
          reinterpret_cast<const unsigned short*>(&xb);
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) s += wf[i] * bf2f(xp[i]);
#pragma unroll
      for (int i = 0; i < 8; ++i) s += wf[8 + i] * bf2f(xq[i]);
      acc[m] += s;
    }
  }
  const float sc = scale[n];
  for (int m = 0; m < M; ++m) {
    float v = wave_reduce_sum(acc[m]) * sc;
    if (lane == 0) {
      if (bias != nullptr) v += bf2f(bias[n]);
      OUT[(long)m * N + n] = f2bf(v);
    }
  }
}

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

extern __shared__ __attribute__((aligned(16))) char smem[];

// 8 fp8 numbers (two words) as bf16
__device__ __forceinline__ bf16x8 gv_widen(int a, int b) {
  i32x4 o;
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    const int v = w ? b : a;
    const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8(v, false);
    const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8(v, true);
    o[w * 2] = __builtin_bit_cast(int, __builtin_convertvector(lo, bf16x2));
    o[w * 2 + 1] =
        __builtin_bit_cast(int, __builtin_convertvector(hi, bf16x2));
  }
  return __builtin_bit_cast(bf16x8, o);
}

// Chunks of a wave's ring: two workgroups share a CU. XR: rows of x staged.
constexpr int gv_ring(bool glu) { return glu ? 3 : 4; }
constexpr int gv_stage(bool glu, int XR) { return (glu ? 4096 : 2048) + XR * 256; }

template <bool GLU, int XR>
__global__ void __launch_bounds__(256)
gemv_fp8_ring_kernel(const unsigned short* __restrict__ X,
                     const unsigned char* __restrict__ W,
                     const float* __restrict__ scale,
                     const unsigned short* __restrict__ bias,
                     unsigned short* __restrict__ OUT, int M, int N, int K) {
  constexpr int NT = GLU ? 2 : 1;
  constexpr int GV_R = gv_ring(GLU), XL = XR / 4;
  constexpr int STAGE = gv_stage(GLU, XR), LOADS = NT * 2 + XL;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int cols = GLU ? N / 2 : N, n0 = blockIdx.x * 16;
  char* ring = smem + wid * GV_R * STAGE;
  // chunks wid, wid + 4, ... from the workgroup's first one on
  const int nch = K / 128, mine = (nch - wid + 3) / 4;
  const int turn = chunk_turn<37>(blockIdx.x, nch) + wid;
  auto chunk = [&](int c) {
    const int k = c * 4 + turn;
    return k >= nch ? k - nch : k;
  };
  const char* src[LOADS];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int row = p * 8 + (lane >> 3);
#pragma unroll
    for (int t = 0; t < NT; ++t)
      src[t * 2 + p] =
          (const char*)W +
          (long)(min(n0 + row, cols - 1) + t * cols) * K +
          ((lane & 7) ^ (row & 7)) * 16;
  }
#pragma unroll
  for (int p = 0; p < XL; ++p) {
    const int row = p * 4 + (lane >> 4);
    src[NT * 2 + p] = (const char*)(X + (long)min(row, M - 1) * K) +
                      ((lane & 15) ^ row) * 16;
  }
  auto issue = [&](int c) {
    char* dst = ring + (c % GV_R) * STAGE + lane * 16;
    const long k = chunk(c) * 128;
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) unsigned int*)(
              src[i] + k * (i < NT * 2 ? 1 : 2)),
          (__attribute__((address_space(3))) unsigned int*)(dst + i * 1024),
          16, 0, 0);
  };
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = {0.f, 0.f, 0.f, 0.f};
  auto compute = [&](int c) {
    const char* b = ring + (c % GV_R) * STAGE;
    const int xr = r & (XR - 1);
    const char* xb = b + NT * 2048 + xr * 256;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      bf16x8 x[2];
#pragma unroll
      for (int e = 0; e < 2; ++e)
        x[e] = *reinterpret_cast<const bf16x8*>(
            xb + (((j * 8 + g * 2 + e) ^ xr) * 16));
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const i32x4 w = *reinterpret_cast<const i32x4*>(
            b + t * 2048 + r * 128 + (((j * 4 + g) ^ (r & 7)) * 16));
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            gv_widen(w[0], w[1]), x[0], acc[t], 0, 0, 0);
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            gv_widen(w[2], w[3]), x[1], acc[t], 0, 0, 0);
      }
    }
    // the buffer is read before the wave fills it again
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  int at = 0;
  while (at < GV_R - 1 && at < mine) issue(at++);
  for (int c = 0; c < mine; ++c) {
    if (at < mine) {
      issue(at++);
      asm volatile("s_waitcnt vmcnt(%0)" ::"i"((GV_R - 1) * LOADS)
                   : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    compute(c);
  }
  __syncthreads();
  float* red = reinterpret_cast<float*>(smem);  // [4][NT][256]
#pragma unroll
  for (int t = 0; t < NT; ++t)
    *reinterpret_cast<f32x4*>(red + (wid * NT + t) * 256 + lane * 4) = acc[t];
  __syncthreads();
  if (threadIdx.x >= 128) return;
  // thread: row m, column n0 + n
  const int m = threadIdx.x >> 4, n = threadIdx.x & 15;
  if (m >= M || n0 + n >= cols) return;
  float v[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    v[t] = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w)
      v[t] += red[(w * NT + t) * 256 + ((n >> 2) * 16 + m) * 4 + (n & 3)];
    v[t] *= scale[n0 + n + t * cols];
    if (bias != nullptr) v[t] += bf2f(bias[n0 + n + t * cols]);
  }
  OUT[(long)m * cols + n0 + n] = f2bf(GLU ? silu(v[0]) * v[NT - 1] : v[0]);
}

// One row with its residual sum and norm ahead (norm_row.h). The normed row
// stays in LDS, the rings hold weights only. In a graph, us, in two launches
// and in one: 28672 x 4096 gated 27.5 and 24.8, 6144 x 4096 10.7 and 8.5 (25.5 and
// 8.7 while the norm waited for the first weights).
constexpr int gv_norm_ring(bool glu) { return glu ? 4 : 6; }
constexpr int gv_norm_lds(bool glu, int K) {
  return 128 + K * 2 + 4 * gv_norm_ring(glu) * (glu ? 4096 : 2048);
}

template <bool GLU, int NC>
__global__ void __launch_bounds__(256)
gemv_fp8_norm_kernel(const NormRow nr, const unsigned char* __restrict__ W,
                     const float* __restrict__ scale,
                     const unsigned short* __restrict__ bias,
                     unsigned short* __restrict__ OUT, int N, int K) {
  constexpr int NT = GLU ? 2 : 1, R = gv_norm_ring(GLU);
  constexpr int STAGE = NT * 2048, LOADS = NT * 2;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int cols = GLU ? N / 2 : N, n0 = blockIdx.x * 16;
  char* hs = smem + 128;
  char* ring = hs + K * 2 + wid * R * STAGE;
  // chunks wid, wid + 4, ... from the workgroup's first one on
  const int nch = K / 128, mine = (nch - wid + 3) / 4;
  const int turn = chunk_turn<37>(blockIdx.x, nch) + wid;
  auto chunk = [&](int c) {
    const int k = c * 4 + turn;
    return k >= nch ? k - nch : k;
  };
  const int rows = min(16, cols - n0);
  int lane_at[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int row = p * 8 + (lane >> 3);
    lane_at[p] = min(row, rows - 1) * K + ((lane & 7) ^ (row & 7)) * 16;
  }
  __amdgpu_buffer_rsrc_t src[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
    src[t] = weight_rows(W + (long)(n0 + t * cols) * K, rows * K);
  auto issue = [&](int c) {
    char* dst = ring + (c % R) * STAGE;
    const int k = chunk(c) * 128;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int p = 0; p < 2; ++p)
        copy_rows_to_lds(src[t], lane_at[p], k, dst + (t * 2 + p) * 1024);
  };
  norm_row<NC>(nr, K, reinterpret_cast<float*>(smem), hs, [&]() {
#pragma unroll
    for (int c = 0; c < R - 1; ++c) issue(c);
  });
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = {0.f, 0.f, 0.f, 0.f};
  auto compute = [&](int c) {
    const char* b = ring + (c % R) * STAGE;
    const char* xb = hs + chunk(c) * 256;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      bf16x8 x[2];
#pragma unroll
      for (int e = 0; e < 2; ++e)
        x[e] = *reinterpret_cast<const bf16x8*>(xb +
                                                (j * 8 + g * 2 + e) * 16);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const i32x4 w = *reinterpret_cast<const i32x4*>(
            b + t * 2048 + r * 128 + (((j * 4 + g) ^ (r & 7)) * 16));
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            gv_widen(w[0], w[1]), x[0], acc[t], 0, 0, 0);
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            gv_widen(w[2], w[3]), x[1], acc[t], 0, 0, 0);
      }
    }
    // the buffer is read before the wave fills it again
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  int c = 0;
  for (; c + R - 1 < mine; ++c) {
    issue(c + R - 1);
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"((R - 1) * LOADS) : "memory");
    compute(c);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  for (; c < mine; ++c) compute(c);
  __syncthreads();
  float* red = reinterpret_cast<float*>(smem);  // [4][NT][256]
#pragma unroll
  for (int t = 0; t < NT; ++t)
    *reinterpret_cast<f32x4*>(red + (wid * NT + t) * 256 + lane * 4) = acc[t];
  __syncthreads();
  const int n = threadIdx.x;  // column n0 + n
  if (n >= 16 || n0 + n >= cols) return;
  float v[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    v[t] = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w)
      v[t] += red[(w * NT + t) * 256 + (n >> 2) * 64 + (n & 3)];
    v[t] *= scale[n0 + n + t * cols];
    if (bias != nullptr) v[t] += bf2f(bias[n0 + n + t * cols]);
  }
  OUT[n0 + n] = f2bf(GLU ? silu(v[0]) * v[NT - 1] : v[0]);
}

// K % 128 == 0 from 2560 (five chunks of 128 for each of four waves) to 8192
extern "C" void launch_gemv_fp8_norm(const void* a, const void* b,
                                     const void* w_norm, void* sum, float eps,
                                     const void* W, const float* scale,
                                     const void* bias, void* out, int N,
                                     int K, bool glu, hipStream_t stream) {
  const NormRow n = {(const unsigned short*)a, (const unsigned short*)b,
                     (const unsigned short*)w_norm, (unsigned short*)sum,
                     eps};
#define GVN(G, NC)                                                          \
  hipLaunchKernelGGL((gemv_fp8_norm_kernel<G, NC>),                         \
                     dim3(((G ? N / 2 : N) + 15) / 16), dim3(256),          \
                     gv_norm_lds(G, K), stream, n, (const unsigned char*)W, \
                     scale, (const unsigned short*)bias,                    \
                     (unsigned short*)out, N, K)
  if (K <= 4096) {
    if (glu) GVN(true, 2);
    else GVN(false, 2);
  } else {
    if (glu) GVN(true, 4);
    else GVN(false, 4);
  }
#undef GVN
}

// glu: W holds gate rows, then up rows; out [M, N / 2]. Needs K % 128 == 0.
extern "C" void launch_gemv_fp8(const void* X, const void* W,
                                const float* scale, const void* bias,
                                void* out, int M, int N, long K, bool glu,
                                hipStream_t stream) {
#define GVR(G, XR)                                                           \
  hipLaunchKernelGGL((gemv_fp8_ring_kernel<G, XR>),                          \
                     dim3(((G ? N / 2 : N) + 15) / 16), dim3(256),           \
                     4 * gv_ring(G) * gv_stage(G, XR), stream,               \
                     (const unsigned short*)X, (const unsigned char*)W,      \
                     scale, (const unsigned short*)bias,                     \
                     (unsigned short*)out, M, N, (int)K)
  if (glu) {
    if (M <= 4) GVR(true, 4);
    else GVR(true, 8);
    return;
  }
  // One row and few columns of a long K: the ring's 16 columns a workgroup leave
  // most CUs without one, a wave per column does not. us, ring and column: 512 x
  // 4096 4.5 and 4.1, x 8192 7.2 and 5.9, x 16384 12.7 and 11.0; 64 x 28672 20.4
  // and 14.4; two rows the same or slower by column.
  if (K % 128 == 0 && !(M == 1 && N <= 512 && K >= 4096)) {
    if (M <= 4) GVR(false, 4);
    else GVR(false, 8);
    return;
  }
#undef GVR
  const int grid = (N + 7) / 8;
  hipLaunchKernelGGL(gemv_fp8_kernel, dim3(grid), dim3(512), 0, stream,
                     (const unsigned short*)X, (const unsigned char*)W,
                     scale, (const unsigned short*)bias,
                     (unsigned short*)out, M, N, K);
}
