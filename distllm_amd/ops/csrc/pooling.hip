// Pooling kernels: masked mean (excl. BOS/EOS) and last-token gather,
// each with fused L2 normalization; fp32 accumulate, fp32 output.
//
// Semantics parity with reference distllm/embed/poolers/mean.py:13-49
// (mask[:,0] and mask[:,L-1] zeroed, clamped count) and
// last_token.py:12-38 (gather at L-1, or S-1 when left-padded), plus the
// F.normalize(p=2) of embedders/full_sequence.py:69 fused in.
#include "common.h"

// hidden [R, S, H] bf16, mask [R, S] int32 -> out [R, H] fp32. Bound by
// reading the unmasked rows. A workgroup has a share of a sequence: its waves
// take every fourth position, four of them in flight, and meet in LDS. With
// few sequences NS workgroups share one and leave sums [R, NS, H] to a second
// launch. 512 x 512 x 768 284 -> 92 us, 32 x 1024 x 1280, half of it masked,
// 330 -> 15 us, by one thread per 8 columns that read position after
// position before.
template <int NCT>  // 8-column pieces of a lane: ceil(H / 512)
__global__ void __launch_bounds__(256)
mean_pool_kernel(const unsigned short* __restrict__ hidden,
                 const int* __restrict__ mask, float* __restrict__ out,
                 float* __restrict__ parts, int R, int S, int H, int NS,
                 bool normalize) {
  extern __shared__ __attribute__((aligned(16))) float sums[];  // [H]
  __shared__ float lds[16];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n_chunks = H >> 3;
  const int split = blockIdx.x % NS, r = blockIdx.x / NS;
  const int* mrow = mask + (long)r * S;

  // row length L = sum(mask[r,:]); of it positions 1 .. L - 2 count (BOS and
  // the last one excluded)
  int lsum = 0;
  for (int s = threadIdx.x; s < S; s += 256) lsum += mrow[s];
  const int L = (int)(block_reduce_sum<4>((float)lsum, lds) + 0.5f);
  const int end = min(L - 1, S), per = (max(end - 1, 0) + NS - 1) / NS;
  const int s0 = 1 + split * per, s1 = min(end, s0 + per);

  float acc[NCT][8];
#pragma unroll
  for (int k = 0; k < NCT; ++k)
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[k][i] = 0.f;
  for (int s = s0 + wid * 4; s < s1; s += 16) {
    s16x8 v[4][NCT];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int k = 0; k < NCT; ++k) {
        const int c = min(lane + k * 64, n_chunks - 1);
        v[j][k] = *reinterpret_cast<const s16x8*>(
            hidden + ((long)r * S + min(s + j, s1 - 1)) * H + c * 8);
      }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // (masks with holes are honored)
      if (s + j >= s1 || !mrow[s + j]) continue;
#pragma unroll
      for (int k = 0; k < NCT; ++k) {
        float f[8];
        bf8_to_f32(v[j][k], f);
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[k][i] += f[i];
      }
    }
  }
  for (int w = 0; w < 4; ++w) {
    if (wid == w) {
#pragma unroll
      for (int k = 0; k < NCT; ++k) {
        const int c = lane + k * 64;
        if (c < n_chunks) {
          float* p = sums + c * 8;
          float f[8];
          if (w > 0) {
            load8(p, f);
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[k][i] += f[i];
          }
          store8(p, acc[k]);
        }
      }
    }
    __syncthreads();
  }
  if (NS > 1) {
    for (int c = threadIdx.x; c < H; c += 256)
      parts[(long)blockIdx.x * H + c] = sums[c];
    return;
  }
  // (a quotient, rounded once; a product with 1 / count is rounded twice more)
  const float count = fmaxf((float)L - 2.f, 1.f);
  float sq = 0.f;
  for (int c = threadIdx.x; c < H; c += 256) {
    const float m = sums[c] / count;
    sums[c] = m;
    sq += m * m;
  }
  const float scale =
      normalize ? rsqrtf(fmaxf(block_reduce_sum<4>(sq, lds), 1e-24f)) : 1.f;
  for (int c = threadIdx.x; c < H; c += 256)
    out[(long)r * H + c] = sums[c] * scale;
}

__global__ void __launch_bounds__(256)
mean_join_kernel(const float* __restrict__ parts, const int* __restrict__ mask,
                 float* __restrict__ out, int S, int H, int NS,
                 bool normalize) {
  extern __shared__ __attribute__((aligned(16))) float sums[];  // [H]
  __shared__ float lds[16];
  const int r = blockIdx.x;
  int lsum = 0;
  for (int s = threadIdx.x; s < S; s += 256) lsum += mask[(long)r * S + s];
  const int L = (int)(block_reduce_sum<4>((float)lsum, lds) + 0.5f);
  const float count = fmaxf((float)L - 2.f, 1.f);
  float sq = 0.f;
  for (int c = threadIdx.x; c < H; c += 256) {
    float m = 0.f;
#pragma unroll 4
    for (int p = 0; p < NS; ++p) m += parts[((long)r * NS + p) * H + c];
    m /= count;
    sums[c] = m;
    sq += m * m;
  }
  const float scale =
      normalize ? rsqrtf(fmaxf(block_reduce_sum<4>(sq, lds), 1e-24f)) : 1.f;
  for (int c = threadIdx.x; c < H; c += 256)
    out[(long)r * H + c] = sums[c] * scale;
}

// last-token gather: out[r,:] = hidden[r, idx, :]; idx = L-1 (right pad)
// or S-1 (left pad); fused L2 normalize.
__global__ void __launch_bounds__(256)
last_token_pool_kernel(const unsigned short* __restrict__ hidden,
                       const int* __restrict__ mask, float* __restrict__ out,
                       int R, int S, int H, bool left_padded, bool normalize) {
  __shared__ float lds[16];
  const int n_chunks = H >> 3;
  for (int r = blockIdx.x; r < R; r += gridDim.x) {
    int idx;
    if (left_padded) {
      idx = S - 1;
    } else {
      int lsum = 0;
      for (int s = threadIdx.x; s < S; s += blockDim.x)
        lsum += mask[r * S + s];
      float L = block_reduce_sum<4>((float)lsum, lds);
      idx = max((int)(L + 0.5f) - 1, 0);
    }
    const unsigned short* hrow = hidden + ((long)r * S + idx) * H;
    float sq = 0.f;
    float vals[8][8];  // up to H=16384
    int nk = (n_chunks + 255) / 256;
#pragma unroll 8
    for (int k = 0; k < nk && k < 8; ++k) {
      const int c = threadIdx.x + k * 256;
      if (c < n_chunks) {
        s16x8 hv = *reinterpret_cast<const s16x8*>(hrow + c * 8);
        bf8_to_f32(hv, vals[k]);
#pragma unroll
        for (int i = 0; i < 8; ++i) sq += vals[k][i] * vals[k][i];
      }
    }
    float scale = 1.f;
    if (normalize) {
      __syncthreads();
      float tot = block_reduce_sum<4>(sq, lds);
      scale = rsqrtf(fmaxf(tot, 1e-24f));
    }
#pragma unroll 8
    for (int k = 0; k < nk && k < 8; ++k) {
      const int c = threadIdx.x + k * 256;
      if (c < n_chunks) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          out[(long)r * H + c * 8 + i] = vals[k][i] * scale;
      }
    }
    __syncthreads();
  }
}

// standalone row-wise L2 normalize, fp32 in/out [R, H]
__global__ void __launch_bounds__(256)
l2_normalize_kernel(const float* __restrict__ x, float* __restrict__ out,
                    int R, int H) {
  __shared__ float lds[16];
  for (int r = blockIdx.x; r < R; r += gridDim.x) {
    float sq = 0.f;
    for (int c = threadIdx.x; c < H; c += blockDim.x) {
      float v = x[(long)r * H + c];
      sq += v * v;
    }
    float tot = block_reduce_sum<4>(sq, lds);
    float scale = rsqrtf(fmaxf(tot, 1e-24f));
    for (int c = threadIdx.x; c < H; c += blockDim.x)
      out[(long)r * H + c] = x[(long)r * H + c] * scale;
    __syncthreads();
  }
}

// Workgroups that share a sequence: two for every CU, each with at least 32
// positions.
extern "C" int mean_pool_shares(int R, int S) {
  return max(min(512 / max(R, 1), S / 32), 1);
}

extern "C" void launch_mean_pool(const void* hidden, const int* mask,
                                 float* out, float* parts, int R, int S,
                                 int H, int NS, bool normalize,
                                 hipStream_t stream) {
  const int nct = (H / 8 + 63) / 64;
#define DM(N)                                                                  \
  hipLaunchKernelGGL((mean_pool_kernel<N>), dim3(R * NS), dim3(256), H * 4,    \
                     stream, (const unsigned short*)hidden, mask, out, parts,  \
                     R, S, H, NS, normalize)
  if (nct <= 1) DM(1);
  else if (nct <= 2) DM(2);
  else if (nct <= 3) DM(3);
  else if (nct <= 4) DM(4);
  else if (nct <= 8) DM(8);
  else if (nct <= 16) DM(16);
  else DM(32);
#undef DM
  if (NS > 1)
    hipLaunchKernelGGL(mean_join_kernel, dim3(R), dim3(256), H * 4, stream,
                       parts, mask, out, S, H, NS, normalize);
}

extern "C" void launch_last_token_pool(const void* hidden, const int* mask,
                                       float* out, int R, int S, int H,
                                       bool left_padded, bool normalize,
                                       hipStream_t stream) {
  hipLaunchKernelGGL(last_token_pool_kernel, dim3(min(R, 2048)), dim3(256), 0,
                     stream, (const unsigned short*)hidden, mask, out, R, S, H,
                     left_padded, normalize);
}

extern "C" void launch_l2_normalize(const float* x, float* out, int R, int H,
                                    hipStream_t stream) {
  hipLaunchKernelGGL(l2_normalize_kernel, dim3(min(R, 2048)), dim3(256), 0,
                     stream, x, out, R, H);
}
