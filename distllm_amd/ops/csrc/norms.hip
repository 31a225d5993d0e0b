// Fused residual + LayerNorm / RMSNorm kernels (bf16 I/O, fp32 math).
//
// Replaces the LayerNorm/RMSNorm work the reference delegated to HF
// transformers model forwards (reference: distllm/embed/encoders/auto.py
// encode() running AutoModel).
//
// Design (guide: Appendix B element-wise/reduction rules):
//  - one WAVE per row (row = hidden vector of size H), 4 rows per 256-thread
//    block; bf16 loads vectorized as s16x8 (16 B/lane);
//  - all that a row needs, weights and bias too, is asked for before its
//    sums: a row's chunks under branches, then its weights, were a round to
//    memory each. Lanes past the row's end ask for its last numbers again
//    (guards instead: 2 to 10% slower). us with a residual, 768 columns,
//    4096 rows 5.9 -> 5.3, 12992 14.0 -> 12.3 (4.9 TB/s), 131072 104 -> 100,
//    262144 205 -> 200 (6.0 TB/s).
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

    s16x8 xv[NCL], rv[NCL], wv[NCL], bv[NCL];
#pragma unroll
    for (int k = 0; k < NCL; ++k) {
      const int c = min(lane + k * WAVE, chunks - 1) * 8;
      xv[k] = *reinterpret_cast<const s16x8*>(xr + c);
      if (HAS_RES) rv[k] = *reinterpret_cast<const s16x8*>(rr + c);
    }
    // The weights behind the row, not ahead of the loop and waited for there, as the
    // compiler would have it up to 512 columns (us then and so, RMS norms of 65536 rows
    // of 128 17.9 and 16.3, with a residual and its sum 26 and 22). Of two and more
    // chunks that is 3 to 5% faster with a sum to write and slower without. The bias,
    // which an RMS norm seldom has, behind its sums: 8192 rows of 640 8.9 and 7.9.
    int behind = 0;
    if (NCL == 1 || WRITE_SUM) asm volatile("" : "+s"(behind));
    auto bias_at = [&](int k) {
      const int c = min(lane + k * WAVE, chunks - 1) * 8 + behind;
      if (b != nullptr) bv[k] = *reinterpret_cast<const s16x8*>(b + c);
      else bv[k] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
    };
#pragma unroll
    for (int k = 0; k < NCL; ++k) {
      const int c = min(lane + k * WAVE, chunks - 1) * 8 + behind;
      wv[k] = *reinterpret_cast<const s16x8*>(w + c);
      if (!RMS) bias_at(k);
    }
    __builtin_amdgcn_sched_barrier(0);

    float v[NCL][8];
    float sum = 0.f, sumsq = 0.f;
#pragma unroll
    for (int k = 0; k < NCL; ++k) {
      const int c = lane + k * WAVE;
      if (c < chunks) {
        float f[8];
        bf8_to_f32(xv[k], f);
        if (HAS_RES) {
          float g[8];
          bf8_to_f32(rv[k], g);
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
        float wf[8], bf[8];
        if (RMS) bias_at(k);
        bf8_to_f32(wv[k], wf);
        bf8_to_f32(bv[k], bf);
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

// ONE 256-thread block per row (4 waves split the chunks, LDS cross-wave
// combine): few rows are a few waves in the kernel above, and wide ones a
// quarter of the waves that a CU could have, for their registers.
// AHEAD: all is asked for at once, as above; else chunk by chunk, and the
// weights behind the sums. us, behind and ahead, with residual and sum: 16
// rows of 4096 2.88 and 2.69, 256 rows of 2048 2.69 and 2.51, 2048 13.8 and
// 13.1 of 4096, 4096 23.6 and 22.5, 13000 rows of 2048 39.2 and 33.1; but
// 800 and 1024 rows of 4096 6.27, 7.00 and 6.56, 7.30, of 1024 2.65, 3.10
// and 2.89, 3.29; 512 rows of 640 to 4096 within 3% either way, 1500 1%.
template <int NCL, bool HAS_RES, bool WRITE_SUM, bool RMS, bool AHEAD>
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

  s16x8 xv[NCL], rv[NCL], wv[NCL], bv[NCL];
  auto row_at = [&](int k) {
    const int c = min((int)threadIdx.x + k * 256, chunks - 1) * 8;
    xv[k] = *reinterpret_cast<const s16x8*>(xr + c);
    if (HAS_RES) rv[k] = *reinterpret_cast<const s16x8*>(rr + c);
  };
  auto weights_at = [&](int k) {
    const int c = min((int)threadIdx.x + k * 256, chunks - 1) * 8;
    wv[k] = *reinterpret_cast<const s16x8*>(w + c);
    if (b != nullptr) bv[k] = *reinterpret_cast<const s16x8*>(b + c);
    else bv[k] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
  };
  if (AHEAD) {
#pragma unroll
    for (int k = 0; k < NCL; ++k) row_at(k);
#pragma unroll
    for (int k = 0; k < NCL; ++k) weights_at(k);
    __builtin_amdgcn_sched_barrier(0);
  }

  float v[NCL][8];
  float sum = 0.f, sumsq = 0.f;
#pragma unroll
  for (int k = 0; k < NCL; ++k) {
    const int c = threadIdx.x + k * 256;
    if (c < chunks) {
      if (!AHEAD) row_at(k);
      float f[8];
      bf8_to_f32(xv[k], f);
      if (HAS_RES) {
        float g[8];
        bf8_to_f32(rv[k], g);
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
      if (!AHEAD) weights_at(k);
      float wf[8], bf[8];
      bf8_to_f32(wv[k], wf);
      bf8_to_f32(bv[k], bf);
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
// threads without any. Measured in a graph with residual (and sum, from 1152
// columns on), us, workgroup and wave per row: 64 rows of 512 2.31 and 2.28, of
// 768 2.34 and 2.54, of 4096 2.8 and 4.5; 2048 rows of 128 3.2 and 2.6, of 512 3.6
// and 3.3, of 768 4.0 and 4.1; 4096 rows of 768 5.7 and 5.3, of 1024 6.4 and 6.1,
// of 1280 8.4 and 8.6, of 2560 15.2 and 17.9; 16384 rows of 768 18.1 and 14.4, of
// 1024 19.6 and 17.9, of 1152 26.7 and 26.7, of 1280 28.4 and 29.4, of 2048 40.7
// and 42.5; 65536 rows of 1152 to 2560 0.95 to 1.01 of the wave's time, 131072
// 0.99 to 1.02; of 4096 always below 0.99. Without a residual 65536 rows of 1152 and
// 1280 70.8 and 64.6, 78.4 and 75.1. With a sum to write 2500 rows of 768 5.7 and 6.1,
// of 1024 6.7 and 7.3, 4096 of 1024 8.6 and 8.6.
static bool norm_row_block(int n_rows, int H, bool has_res, bool write_sum) {
  const int narrow = write_sum && H > 640 ? 3000 : 2048;
  const int wide = has_res || H >= 1536 ? 65536 : 16384;
  return n_rows <= 8 || (H > 512 && n_rows <= narrow) ||
         (H > 1024 && n_rows <= wide) || H >= 3072;
}

extern "C" void launch_norm_fwd(const void* x, const void* res, const void* w,
                                const void* b, void* out, void* sum_out,
                                int n_rows, int H, float eps, bool rms,
                                hipStream_t stream) {
  // Waves that go on to a second row pay up to 512 columns only: us, at most
  // 32768 blocks and all, 262144 rows of 128 50.7 and 63.6, of 384 102.8 and
  // 105.8, of 768 209 and 200, of 1024 281 and 278, of 1280 466 and 455, of 2048
  // 763 and 749. (Threads of a grid are counted in 32 bits: at most 2^20 blocks.)
  static const int cap = [] {
    const char* e = getenv("DISTLLM_NORM_BLOCKS");
    return e ? atoi(e) : 0;
  }();
  int blocks = min((n_rows + 3) / 4,
                   cap != 0 ? cap : H > 512 ? 1 << 20 : 32768);
  bool has_res = res != nullptr;
  bool write_sum = sum_out != nullptr;
  const bool small = norm_row_block(n_rows, H, has_res, write_sum);
  // (2048 rows without a residual: of 640 and 768 columns 3.88 ahead and 3.70, of 8192
  // 16.2 and 14.4)
  const bool ahead =
      n_rows <= 512 || n_rows > 2048 ||
      (n_rows >= 1500 && H > 1024 && (has_res || H < 3072));
  int ncl = small ? (H / 8 + 255) / 256 : (H / 8 + WAVE - 1) / WAVE;

#define DISPATCH4(KERNEL, BLOCKS)                                              \
  hipLaunchKernelGGL(KERNEL, dim3(BLOCKS), dim3(256), 0, stream,               \
                     (const unsigned short*)x, (const unsigned short*)res,     \
                     (const unsigned short*)w, (const unsigned short*)b,       \
                     (unsigned short*)out, (unsigned short*)sum_out, n_rows,   \
                     H, eps)
#define DISPATCH3(NCL, HR, WS, RM)                                             \
  do {                                                                         \
    if (small && ahead)                                                        \
      DISPATCH4((norm_fwd_small_kernel<NCL, HR, WS, RM, true>), n_rows);       \
    else if (small)                                                            \
      DISPATCH4((norm_fwd_small_kernel<NCL, HR, WS, RM, false>), n_rows);      \
    else                                                                       \
      DISPATCH4((norm_fwd_kernel<NCL, HR, WS, RM>), blocks);                   \
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
#undef DISPATCH4
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
