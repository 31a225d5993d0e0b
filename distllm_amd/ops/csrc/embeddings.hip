// Start of a BERT-class encoder: out = layer norm of word[id] + pos[p] +
// type, one launch for a gather, two additions and the norm, which each wrote
// the whole [tokens, H] in bf16; and the additive key mask of the attention.
// Bound by the gathered rows and the output (both once): 512 x 512 tokens of
// 768, 610 -> 175 us. A wave per token. What does not come by the token's number (type
// row, weights, bias, rows of positions that are counted) is asked for ahead of it, up
// to 2048 columns, and the mask goes along: few tokens are a chain of rounds to memory,
// and a launch of its own for the mask is one more. 24 tokens of 768 5.0 -> 4.3 us under
// the profiler, an encoder of 12 layers on them 288 -> 286.
#include "common.h"

// Row of a table of n, from the end if negative; as torch's indexing, a number
// outside the table ends the program.
__device__ __forceinline__ long table_row(long i, long n) {
  if (i < 0) i += n;
  if (i < 0 || i >= n) __builtin_trap();
  return i;
}

template <int NCL>  // 8-column pieces of a lane
__global__ void __launch_bounds__(256)
embed_layer_norm_kernel(const long* __restrict__ ids,
                        const long* __restrict__ pos_ids,
                        const unsigned short* __restrict__ word,
                        const unsigned short* __restrict__ pos,
                        const unsigned short* __restrict__ type,
                        const unsigned short* __restrict__ w,
                        const unsigned short* __restrict__ b,
                        unsigned short* __restrict__ out, long n_rows, int S,
                        int H, long n_words, long n_pos, float eps,
                        const void* __restrict__ mask, int mask_bytes,
                        float* __restrict__ key_bias) {
  const int lane = threadIdx.x & 63;
  const long row = (long)blockIdx.x * 4 +
                   __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (row >= n_rows) return;
  const int chunks = H >> 3;
  constexpr bool AHEAD = NCL <= 4;
  constexpr int HELD = AHEAD ? NCL : 1;
  s16x8 held[3][HELD];
  if (AHEAD) {
#pragma unroll
    for (int k = 0; k < NCL; ++k) {
      const int c = min(lane + k * 64, chunks - 1) * 8;
      held[0][k] = *reinterpret_cast<const s16x8*>(type + c);
      held[1][k] = *reinterpret_cast<const s16x8*>(w + c);
      held[2][k] = *reinterpret_cast<const s16x8*>(b + c);
    }
  }
  auto shared8 = [&](int which, const unsigned short* from, int k, int c,
                     float* f) {
    if (AHEAD) bf8_to_f32(held[which][AHEAD ? k : 0], f);
    else load8(from + c * 8, f);
  };
  const unsigned short* a = word + table_row(ids[row], n_words) * H;
  const unsigned short* p =
      pos +
      (pos_ids != nullptr ? table_row(pos_ids[row], n_pos) : row % S) * H;
  if (mask_bytes != 0 && lane == 0)
    key_bias[row] = (mask_bytes == 1 ? static_cast<const char*>(mask)[row] != 0
                     : mask_bytes == 4
                         ? static_cast<const int*>(mask)[row] != 0
                         : static_cast<const long*>(mask)[row] != 0)
                        ? 0.f
                        : -INFINITY;
  float v[NCL][8];
  float sum = 0.f, sumsq = 0.f;
#pragma unroll
  for (int k = 0; k < NCL; ++k) {
    const int c = lane + k * 64;
    if (c < chunks) {
      float f[8], t[8];
      load8(a + c * 8, v[k]);
      load8(p + c * 8, f);
      shared8(0, type, k, c, t);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[k][i] += f[i] + t[i];
        sum += v[k][i];
        sumsq += v[k][i] * v[k][i];
      }
    }
  }
  sum = wave_reduce_sum(sum);
  sumsq = wave_reduce_sum(sumsq);
  const float mean = sum / H;
  const float inv = rsqrtf(fmaxf(sumsq / H - mean * mean, 0.f) + eps);
#pragma unroll
  for (int k = 0; k < NCL; ++k) {
    const int c = lane + k * 64;
    if (c < chunks) {
      float f[8], t[8];
      shared8(1, w, k, c, f);
      shared8(2, b, k, c, t);
#pragma unroll
      for (int i = 0; i < 8; ++i) f[i] = (v[k][i] - mean) * inv * f[i] + t[i];
      store8(out + row * H + c * 8, f);
    }
  }
}

extern "C" void launch_embed_layer_norm(const long* ids, const long* pos_ids,
                                        const void* word, const void* pos,
                                        const void* type, const void* w,
                                        const void* b, void* out, long n_rows,
                                        int S, int H, long n_words,
                                        long n_pos, float eps,
                                        const void* mask, int mask_bytes,
                                        float* key_bias,
                                        hipStream_t stream) {
  const int ncl = (H / 8 + 63) / 64;
#define EL(N)                                                              \
  hipLaunchKernelGGL(embed_layer_norm_kernel<N>, dim3((n_rows + 3) / 4),   \
                     dim3(256), 0, stream, ids, pos_ids,                   \
                     (const unsigned short*)word,                          \
                     (const unsigned short*)pos,                           \
                     (const unsigned short*)type, (const unsigned short*)w, \
                     (const unsigned short*)b, (unsigned short*)out,       \
                     n_rows, S, H, n_words, n_pos, eps, mask, mask_bytes,  \
                     key_bias)
  if (ncl <= 1) EL(1);
  else if (ncl <= 2) EL(2);
  else if (ncl <= 4) EL(4);
  else if (ncl <= 8) EL(8);
  else EL(16);
#undef EL
}

// 0 where the mask is not zero, -inf where it is
template <typename T>
__global__ void __launch_bounds__(256)
key_bias_kernel(const T* __restrict__ mask, float* __restrict__ out, long n) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = mask[i] != 0 ? 0.f : -INFINITY;
}

extern "C" void launch_key_bias(const void* mask, float* out, long n,
                                int bytes, hipStream_t stream) {
  const dim3 grid((n + 255) / 256);
  if (bytes == 1)
    hipLaunchKernelGGL(key_bias_kernel<signed char>, grid, dim3(256), 0,
                       stream, (const signed char*)mask, out, n);
  else if (bytes == 4)
    hipLaunchKernelGGL(key_bias_kernel<int>, grid, dim3(256), 0, stream,
                       (const int*)mask, out, n);
  else
    hipLaunchKernelGGL(key_bias_kernel<long>, grid, dim3(256), 0, stream,
                       (const long*)mask, out, n);
}
