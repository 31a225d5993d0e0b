// RoPE (rotary position embedding) application, half-split (NeoX) style:
//   out[..., :D/2] = x1*cos - x2*sin ; out[..., D/2:] = x2*cos + x1*sin
// used by Mistral/Llama and ESM2 (K3).
//
// cos/sin tables are HOST-precomputed f32 [S, D/2] (guide Appendix B:
// on-device trig turns memory-bound into VALU-bound).
// x: [B, S, Hx, D] bf16, in-place or out-of-place; pos gives the
// absolute position of each token row (int32 [B, S]) so the same kernel
// serves prefill (pos = arange) and decode (pos = context offsets).
#include "common.h"

__global__ void __launch_bounds__(256)
rope_kernel(const unsigned short* __restrict__ x,
            unsigned short* __restrict__ out,
            const float* __restrict__ cs,   // [max_pos, D/2] cos
            const float* __restrict__ sn,   // [max_pos, D/2] sin
            const int* __restrict__ pos,    // [B*S] absolute positions
            long n_rows,                    // B*S*Hx
            int Hx, int D, int rope_heads) {
  // heads >= rope_heads pass through unchanged: lets ONE launch rope
  // the q|k part of a fused qkv tensor while copying v (decode-path
  // launch fusion)
  const int half = D / 2;
  const long stride = (long)gridDim.x * blockDim.x;
  const long total = n_rows * half;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += stride) {
    const long row = i / half;
    const int d = (int)(i % half);
    const long tok = row / Hx;
    if ((int)(row - tok * Hx) >= rope_heads) {
      const unsigned short* xr = x + row * D;
      out[row * D + d] = xr[d];
      out[row * D + d + half] = xr[d + half];
      continue;
    }
    const int p = pos[tok];
    const float c = cs[(long)p * half + d];
    const float s = sn[(long)p * half + d];
    const unsigned short* xr = x + row * D;
    float x1 = bf2f(xr[d]);
    float x2 = bf2f(xr[d + half]);
    out[row * D + d] = f2bf(x1 * c - x2 * s);
    out[row * D + d + half] = f2bf(x2 * c + x1 * s);
  }
}

extern "C" void launch_rope(const void* x, void* out, const float* cs,
                            const float* sn, const int* pos, long n_rows,
                            int Hx, int D, int rope_heads,
                            hipStream_t stream) {
  const long total = n_rows * (D / 2);
  int blocks = (int)min((total + 255) / 256, (long)2048);
  hipLaunchKernelGGL(rope_kernel, dim3(blocks), dim3(256), 0, stream,
                     (const unsigned short*)x, (unsigned short*)out, cs, sn,
                     pos, n_rows, Hx, D, rope_heads);
}

// The same in place for the first `heads` of the Hx heads of every row, rows
// ld numbers apart: what lies behind them (values beside queries and keys)
// stays where it is. A thread has 8 columns of both halves and loops over
// heads with its part of the table in registers; 8 heads of a row side by
// side. Bound by reading and writing the rotated heads: 16384 rows of 40 heads
// of 128 (of 48) 172 us by the kernel above, which copies all 48 two bytes at
// a time, -> 53 us; 17664 rows of 40 heads of 64 68 us in two calls of that,
// after two copies of 19 us, -> 37 us.
template <int D>
__global__ void __launch_bounds__(256)
rope_inplace_kernel(unsigned short* __restrict__ x,
                    const float* __restrict__ cs,
                    const float* __restrict__ sn,
                    const int* __restrict__ pos, long n_rows, long ld,
                    int heads) {
  constexpr int PER = D / 16;            // threads of a head
  constexpr int ROWS = 256 / (PER * 8);  // rows of a workgroup
  const int c = threadIdx.x % PER * 8;
  const int h0 = threadIdx.x / PER % 8;
  const long row = (long)blockIdx.x * ROWS + threadIdx.x / (PER * 8);
  if (row >= n_rows) return;
  const long t = (long)pos[row] * (D / 2) + c;
  float co[8], si[8];
  load8(cs + t, co);
  load8(sn + t, si);
  for (int h = h0; h < heads; h += 8) {
    unsigned short* p = x + row * ld + (long)h * D + c;
    float a[8], b[8], o[8];
    load8(p, a);
    load8(p + D / 2, b);
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = a[i] * co[i] - b[i] * si[i];
    store8(p, o);
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = b[i] * co[i] + a[i] * si[i];
    store8(p + D / 2, o);
  }
}

extern "C" void launch_rope_inplace(void* x, const float* cs, const float* sn,
                                    const int* pos, long n_rows, long ld,
                                    int heads, int D, hipStream_t stream) {
#define RI(DD)                                                              \
  hipLaunchKernelGGL(rope_inplace_kernel<DD>,                               \
                     dim3((n_rows * (DD / 16) * 8 + 255) / 256), dim3(256), \
                     0, stream, (unsigned short*)x, cs, sn, pos, n_rows, ld, \
                     heads)
  if (D == 64) RI(64);
  else RI(128);
#undef RI
}
