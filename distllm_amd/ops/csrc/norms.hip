// Fused residual + LayerNorm / RMSNorm kernels (bf16 I/O, fp32 math).
//
// Replaces the LayerNorm/RMSNorm work the reference delegated to HF
// transformers model forwards (reference: distllm/embed/encoders/auto.py
// encode() running AutoModel).
//
// Design (guide: Appendix B element-wise/reduction rules):
//  - one WAVE per row (row = hidden vector of size H), 4 rows per 256-thread
//    block; bf16 loads vectorized as s16x8 (16 B/lane);
//  - fp32 accumulate, single pass, row held in registers. Per-lane chunk
//    count is a template parameter so every register index is
//    compile-time (runtime-indexed ext_vector arrays spill to scratch).
//  - optional residual add fused, optional write-back of the summed
//    residual stream (pre-norm architectures need it for the next skip).
#include "common.h"

template <int NCL, bool HAS_RES, bool WRITE_SUM, bool RMS>
__global__ void __launch_bounds__(256)
norm_fwd_kernel(const unsigned short* __restrict__ x,
                const unsigned short* __restrict__ res,
                const unsigned short* __restrict__ w,
                const unsigned short* __restrict__ b,
                unsigned short* __restrict__ out,
                unsigned short* __restrict__ sum_out,
                int n_rows, int H, float eps) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = threadIdx.x >> 6;
  const int waves_per_grid = (gridDim.x * blockDim.x) >> 6;
  const int chunks = H >> 3;  // H multiple of 8 enforced host-side

  for (int row = blockIdx.x * 4 + wid; row < n_rows; row += waves_per_grid) {
    const unsigned short* xr = x + (long)row * H;
    const unsigned short* rr = HAS_RES ? res + (long)row * H : nullptr;

    float v[NCL][8];
    float sum = 0.f, sumsq = 0.f;
#pragma unroll
    for (int k = 0; k < NCL; ++k) {
      const int c = lane + k * WAVE;
      if (c < chunks) {
        s16x8 xv = *reinterpret_cast<const s16x8*>(xr + c * 8);
        float f[8];
        bf8_to_f32(xv, f);
        if (HAS_RES) {
          s16x8 rv = *reinterpret_cast<const s16x8*>(rr + c * 8);
          float g[8];
          bf8_to_f32(rv, g);
#pragma unroll
          for (int i = 0; i < 8; ++i) f[i] += g[i];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          v[k][i] = f[i];
          sum += f[i];
          sumsq += f[i] * f[i];
        }
        if (WRITE_SUM) {
          s16x8 sv;
#pragma unroll
          for (int i = 0; i < 8; ++i) sv[i] = (short)f2bf(f[i]);
          *reinterpret_cast<s16x8*>(sum_out + (long)row * H + c * 8) = sv;
        }
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[k][i] = 0.f;
      }
    }
    sum = wave_reduce_sum(sum);
    sumsq = wave_reduce_sum(sumsq);
    float mean, inv;
    if (RMS) {
      mean = 0.f;
      inv = rsqrtf(sumsq / H + eps);
    } else {
      mean = sum / H;
      inv = rsqrtf(fmaxf(sumsq / H - mean * mean, 0.f) + eps);
    }
#pragma unroll
    for (int k = 0; k < NCL; ++k) {
      const int c = lane + k * WAVE;
      if (c < chunks) {
        s16x8 wv = *reinterpret_cast<const s16x8*>(w + c * 8);
        float wf[8];
        bf8_to_f32(wv, wf);
        float bf[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        if (b != nullptr) {
          s16x8 bv = *reinterpret_cast<const s16x8*>(b + c * 8);
          bf8_to_f32(bv, bf);
        }
        s16x8 ov;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          float y = (v[k][i] - mean) * inv * wf[i] + bf[i];
          ov[i] = (short)f2bf(y);
        }
        *reinterpret_cast<s16x8*>(out + (long)row * H + c * 8) = ov;
      }
    }
  }
}



// Small-batch variant: ONE 256-thread block per row (4 waves split the
// chunks, LDS cross-wave combine). With few rows the wave-per-row kernel is
// a few waves doing NCL dependent 16-B load rounds; spreading the row across
// the block quarters the rounds on the per-token critical path.
template <int NCL, bool HAS_RES, bool WRITE_SUM, bool RMS>
__global__ void __launch_bounds__(256)
norm_fwd_small_kernel(const unsigned short* __restrict__ x,
                      const unsigned short* __restrict__ res,
                      const unsigned short* __restrict__ w,
                      const unsigned short* __restrict__ b,
                      unsigned short* __restrict__ out,
                      unsigned short* __restrict__ sum_out,
                      int n_rows, int H, float eps) {
  __shared__ float red[8];
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = threadIdx.x >> 6;
  const int chunks = H >> 3;
  const int row = blockIdx.x;
  if (row >= n_rows) return;
  const unsigned short* xr = x + (long)row * H;
  const unsigned short* rr = HAS_RES ? res + (long)row * H : nullptr;

  float v[NCL][8];
  float sum = 0.f, sumsq = 0.f;
#pragma unroll
  for (int k = 0; k < NCL; ++k) {
    const int c = threadIdx.x + k * 256;
    if (c < chunks) {
      s16x8 xv = *reinterpret_cast<const s16x8*>(xr + c * 8);
      float f[8];
      bf8_to_f32(xv, f);
      if (HAS_RES) {
        s16x8 rv = *reinterpret_cast<const s16x8*>(rr + c * 8);
        float g[8];
        bf8_to_f32(rv, g);
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] += g[i];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[k][i] = f[i];
        sum += f[i];
        sumsq += f[i] * f[i];
      }
      if (WRITE_SUM) {
        s16x8 sv;
#pragma unroll
        for (int i = 0; i < 8; ++i) sv[i] = (short)f2bf(f[i]);
        *reinterpret_cast<s16x8*>(sum_out + (long)row * H + c * 8) = sv;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[k][i] = 0.f;
    }
  }
  sum = wave_reduce_sum(sum);
  sumsq = wave_reduce_sum(sumsq);
  if (lane == 0) { red[wid] = sum; red[4 + wid] = sumsq; }
  __syncthreads();
  sum = red[0] + red[1] + red[2] + red[3];
  sumsq = red[4] + red[5] + red[6] + red[7];
  float mean, inv;
  if (RMS) {
    mean = 0.f;
    inv = rsqrtf(sumsq / H + eps);
  } else {
    mean = sum / H;
    inv = rsqrtf(fmaxf(sumsq / H - mean * mean, 0.f) + eps);
  }
#pragma unroll
  for (int k = 0; k < NCL; ++k) {
    const int c = threadIdx.x + k * 256;
    if (c < chunks) {
      s16x8 wv = *reinterpret_cast<const s16x8*>(w + c * 8);
      float wf[8];
      bf8_to_f32(wv, wf);
      float bf[8] = {0, 0, 0, 0, 0, 0, 0, 0};
      if (b != nullptr) {
        s16x8 bv = *reinterpret_cast<const s16x8*>(b + c * 8);
        bf8_to_f32(bv, bf);
      }
      s16x8 ov;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float y = (v[k][i] - mean) * inv * wf[i] + bf[i];
        ov[i] = (short)f2bf(y);
      }
      *reinterpret_cast<s16x8*>(out + (long)row * H + c * 8) = ov;
    }
  }
}

// Whether a row gets a workgroup: few rows leave most CUs without a wave, wide
// rows leave a wave with many loads; narrow ones leave most of a workgroup's
// threads without any. Measured in a graph with residual and sum, us, workgroup
// and wave per row: 64 rows of 768 2.6 and 3.3, of 4096 3.4 and 6.6, of 8192
// 4.6 and 11.1; 2048 rows of 128 3.1 and 2.4, of 512 3.4 and 2.8, of 640 1.03
// times the wave's, of 768 4.2 and 4.3, of 4096 9.2 and 11.5, of 8192 15.7 and
// 20.4; 4096 rows of 768 6.4 and 5.5, of 4096 16.1 and 20.7, of 8192 30.3 and
// 37.9. Widths up to 512 are within 4% of each other up to 1024 rows; 3072 to
// 65536 rows of 2048 are 0.91 to 1.14 of the wave's time, of 3072 0.87 to 1.00,
// of 4096 0.83 to 0.96, of 5120 and 8192 0.79 to 0.92.
static bool norm_row_block(int n_rows, int H) {
  return n_rows <= 8 || (H > 512 && n_rows <= 2048) || H >= 3072;
}

extern "C" void launch_norm_fwd(const void* x, const void* res, const void* w,
                                const void* b, void* out, void* sum_out,
                                int n_rows, int H, float eps, bool rms,
                                hipStream_t stream) {
  // Grid cap: measured on MI355X (DISTLLM_NORM_BLOCKS sweep in
  // profiles/RESULTS.md): deep grids beat a 2048-block grid-stride
  // loop by ~5%; a 2-rows-per-wave ILP variant was also probed and
  // REGRESSED (149 -> 172 us plain LN) — tail guards in the unrolled
  // loops cost more than the overlap wins, so R stays 1.
  static const int cap = [] {
    const char* e = getenv("DISTLLM_NORM_BLOCKS");
    return e ? atoi(e) : 32768;
  }();
  int blocks = min((n_rows + 3) / 4, cap);
  bool has_res = res != nullptr;
  bool write_sum = sum_out != nullptr;
  const bool small = norm_row_block(n_rows, H);
  int ncl = small ? (H / 8 + 255) / 256 : (H / 8 + WAVE - 1) / WAVE;

#define DISPATCH3(NCL, HR, WS, RM)                                             \
  do {                                                                         \
    if (small)                                                                 \
      hipLaunchKernelGGL((norm_fwd_small_kernel<NCL, HR, WS, RM>),             \
                         dim3(n_rows), dim3(256), 0, stream,                   \
                         (const unsigned short*)x,                             \
                         (const unsigned short*)res,                           \
                         (const unsigned short*)w,                             \
                         (const unsigned short*)b, (unsigned short*)out,       \
                         (unsigned short*)sum_out, n_rows, H, eps);            \
    else                                                                       \
      hipLaunchKernelGGL((norm_fwd_kernel<NCL, HR, WS, RM>), dim3(blocks),     \
                         dim3(256), 0, stream, (const unsigned short*)x,       \
                         (const unsigned short*)res,                           \
                         (const unsigned short*)w,                             \
                         (const unsigned short*)b, (unsigned short*)out,       \
                         (unsigned short*)sum_out, n_rows, H, eps);            \
  } while (0)
#define DISPATCH_FLAGS(NCL)                                                    \
  do {                                                                         \
    if (rms) {                                                                 \
      if (has_res && write_sum) DISPATCH3(NCL, true, true, true);              \
      else if (has_res) DISPATCH3(NCL, true, false, true);                     \
      else DISPATCH3(NCL, false, false, true);                                 \
    } else {                                                                   \
      if (has_res && write_sum) DISPATCH3(NCL, true, true, false);             \
      else if (has_res) DISPATCH3(NCL, true, false, false);                    \
      else DISPATCH3(NCL, false, false, false);                                \
    }                                                                          \
  } while (0)

  switch (ncl) {
    case 1: DISPATCH_FLAGS(1); break;
    case 2: DISPATCH_FLAGS(2); break;
    case 3: DISPATCH_FLAGS(3); break;
    case 4: DISPATCH_FLAGS(4); break;
    case 5: case 6: DISPATCH_FLAGS(6); break;
    case 7: case 8: DISPATCH_FLAGS(8); break;
    default: DISPATCH_FLAGS(16); break;  // up to H=8192
  }
#undef DISPATCH_FLAGS
#undef DISPATCH3
}

// Sum of the fp32 slabs [S, rows, H] of a product whose K was shared, rounded
// to bf16 as the product would be, + res -> sum_out, and its RMS norm -> out.
// 512 threads a row, all slabs' loads in flight: as many rows as a decode
// step has leave the CUs to latency. With the summing kernel as a launch of
// its own, product and norm in a graph, us: 64 rows 4096 x 14336 33.4 -> 28.8,
// 4096 x 4096 14.9 -> 11.9; 17 rows 4096 x 14336 28.5 -> 25.1.
template <int NCL>
__global__ void __launch_bounds__(512)
norm_parts_kernel(const float* __restrict__ parts, int S,
                  const unsigned short* __restrict__ res,
                  const unsigned short* __restrict__ w,
                  unsigned short* __restrict__ out,
                  unsigned short* __restrict__ sum_out, int n_rows, int H,
                  float eps) {
  __shared__ float red[8];
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = threadIdx.x >> 6;
  const long row = (long)blockIdx.x * H;
  const long slab = (long)n_rows * H;
  float v[NCL][8];
  float sumsq = 0.f;
#pragma unroll
  for (int k = 0; k < NCL; ++k) {
    const int c = (threadIdx.x + k * 512) * 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[k][i] = 0.f;
    if (c < H) {
      const s16x8 rv = *reinterpret_cast<const s16x8*>(res + row + c);
#pragma unroll 4
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4 p = *reinterpret_cast<const f32x4*>(
              parts + s * slab + row + c + h * 4);
#pragma unroll
          for (int i = 0; i < 4; ++i) v[k][h * 4 + i] += p[i];
        }
      float g[8];
      bf8_to_f32(rv, g);
      s16x8 sv;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[k][i] = bf2f(f2bf(v[k][i])) + g[i];
        sumsq += v[k][i] * v[k][i];
        sv[i] = (short)f2bf(v[k][i]);
      }
      *reinterpret_cast<s16x8*>(sum_out + row + c) = sv;
    }
  }
  sumsq = wave_reduce_sum(sumsq);
  if (lane == 0) red[wid] = sumsq;
  __syncthreads();
  sumsq = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) sumsq += red[i];
  const float inv = rsqrtf(sumsq / H + eps);
#pragma unroll
  for (int k = 0; k < NCL; ++k) {
    const int c = (threadIdx.x + k * 512) * 8;
    if (c < H) {
      float wf[8];
      bf8_to_f32(*reinterpret_cast<const s16x8*>(w + c), wf);
      s16x8 ov;
#pragma unroll
      for (int i = 0; i < 8; ++i) ov[i] = (short)f2bf(v[k][i] * inv * wf[i]);
      *reinterpret_cast<s16x8*>(out + row + c) = ov;
    }
  }
}

extern "C" void launch_norm_parts(const float* parts, int S, const void* res,
                                  const void* w, void* out, void* sum_out,
                                  int n_rows, int H, float eps,
                                  hipStream_t stream) {
#define NP(NCL)                                                              \
  hipLaunchKernelGGL(norm_parts_kernel<NCL>, dim3(n_rows), dim3(512), 0,     \
                     stream, parts, S, (const unsigned short*)res,           \
                     (const unsigned short*)w, (unsigned short*)out,         \
                     (unsigned short*)sum_out, n_rows, H, eps)
  if (H <= 4096) NP(1);
  else NP(2);  // up to 8192
#undef NP
}
