// Common device helpers for distllm-amd CDNA4 (gfx950) kernels.
// Hardware model per /opt/skills/guides/cdna_hip_programming.md:
//   wave = 64 lanes, 4 SIMD-32/CU, 160 KiB LDS/CU, MFMA bf16 K=16/32.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>

#define WAVE 64

// ---- vector types -------------------------------------------------------
typedef __attribute__((ext_vector_type(2))) float  f32x2;
typedef __attribute__((ext_vector_type(4))) float  f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) short  s16x4;
typedef __attribute__((ext_vector_type(8))) short  s16x8;
typedef __attribute__((ext_vector_type(2))) int    i32x2;
typedef __attribute__((ext_vector_type(4))) int    i32x4;

// bf16 <-> f32 (scalar); use __hip_bfloat16 for storage only.
__device__ __forceinline__ float bf2f(unsigned short u) {
  union { float f; unsigned int i; } c;
  c.i = ((unsigned int)u) << 16;
  return c.f;
}
__device__ __forceinline__ unsigned short f2bf(float f) {
  // hardware RTNE converter (v_cvt_*_bf16_f32 on gfx950) — far cheaper
  // than the 5-op manual rounding sequence.
  __bf16 h = (__bf16)f;
  union { __bf16 h; unsigned short u; } c;
  c.h = h;
  return c.u;
}

// Convert 8 bf16 (s16x8) to 8 f32.
__device__ __forceinline__ void bf8_to_f32(const s16x8 v, float* out) {
#pragma unroll
  for (int i = 0; i < 8; ++i) out[i] = bf2f((unsigned short)v[i]);
}

// ---- wave reductions (64-wide) -----------------------------------------
// f(v, v of the lane 32 or 16 on or back), by a swap of lanes: on the vector units,
// where __shfl_xor goes through LDS. All lanes of the wave have to be there.
template <int APART, class F>
__device__ __forceinline__ float lanes_join(float v, F f) {
  static_assert(APART == 32 || APART == 16, "halves or quarters");
  const int i = __builtin_bit_cast(int, v);
  const i32x2 s = APART == 32
                      ? __builtin_amdgcn_permlane32_swap(i, i, false, false)
                      : __builtin_amdgcn_permlane16_swap(i, i, false, false);
  const int a = s[0], b = s[1];  // a cast of s[1] itself takes s[0]
  return f(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
}
template <int APART>
__device__ __forceinline__ float lanes_sum(float v) {
  return lanes_join<APART>(v, [](float a, float b) { return a + b; });
}
template <int APART>
__device__ __forceinline__ float lanes_max(float v) {
  return lanes_join<APART>(v, [](float a, float b) { return fmaxf(a, b); });
}
// v of the lane APART back in the ring of 16 that a lane is in
template <int APART>
__device__ __forceinline__ float lane_turned(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v),
                                         0x120 + APART, 0xf, 0xf, false));
}
// Lanes 32, 16, 8, 4, 2, 1 apart are joined; a turn reaches the lane that an XOR
// would, or one of the same sum. Six steps through LDS are a chain of some 0.2 us,
// which kernels of few rows wait for: a step of 32 rows through eight layers of
// latent attention 1318 -> 1303 us, one row's with 8-bit weights 570 -> 568.
__device__ __forceinline__ float wave_reduce_sum(float v) {
  v = lanes_sum<16>(lanes_sum<32>(v));
  v += lane_turned<8>(v);
  v += lane_turned<4>(v);
  v += lane_turned<2>(v);
  v += lane_turned<1>(v);
  return v;
}
__device__ __forceinline__ float wave_reduce_max(float v) {
  v = lanes_max<16>(lanes_max<32>(v));
  v = fmaxf(v, lane_turned<8>(v));
  v = fmaxf(v, lane_turned<4>(v));
  v = fmaxf(v, lane_turned<2>(v));
  v = fmaxf(v, lane_turned<1>(v));
  return v;
}

// Order one wave's LDS accesses across its lanes.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The leading 8 bits of a and b, not negative, as bf16 numbers (a's in the low
// half); a and b become what is left of them, or the least normal number where
// nothing is, which counts for nothing in a sum but keeps a product with infinity
// from being NaN.
__device__ __forceinline__ unsigned int split_bf16(float& a, float& b) {
  const unsigned int h = __builtin_amdgcn_perm(
      __builtin_bit_cast(unsigned int, b), __builtin_bit_cast(unsigned int, a),
      0x07060302);
  a = fmaxf(a - __builtin_bit_cast(float, h << 16), 0x1p-126f);
  b = fmaxf(b - __builtin_bit_cast(float, h & 0xffff0000u), 0x1p-126f);
  return h;
}

// 16 or 4 bytes a lane from global memory to LDS: lane i's to base + i times
// as many, base the same for the whole wave. In assembly, for the compiler
// must not know of it: it lets a transposing read of LDS (ds_read_b64_tr_b16)
// wait for every copy that it knows to be in flight, also those into other
// buffers. So nothing waits by itself, __syncthreads() neither: the caller
// counts its copies and waits (s_waitcnt vmcnt) before a barrier or a read of
// the bytes. M0 is reserved: the compiler sets it ahead of each of its own uses
// and neither keeps nor expects anything in it across assembly, for which a
// clobber would do nothing but warn. (Copies by the builtin would be such uses;
// the kernels that take this have none.)
template <int BYTES = 16>
__device__ __forceinline__ void copy_to_lds(const void* src,
                                            const void* base) {
  const unsigned int at = __builtin_amdgcn_readfirstlane(
      (unsigned int)(uintptr_t)(const __attribute__((address_space(3)))
                                    char*)base);
  static_assert(BYTES == 16 || BYTES == 4, "a copy's width");
  if constexpr (BYTES == 16)
    asm volatile(
        "s_mov_b32 m0, %0\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, off"
        :
        : "s"(at), "v"(src)
        : "memory");
  else
    asm volatile(
        "s_mov_b32 m0, %0\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dword %1, off"
        :
        : "s"(at), "v"(src)
        : "memory");
}

// The same from a pointer that all lanes share, to byte `at` of LDS on.
__device__ __forceinline__ void copy_to_lds(const void* from,
                                            unsigned int lane_at,
                                            unsigned int at) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %2"
      :
      : "s"(at), "v"(lane_at), "s"(from)
      : "memory");
}

// The same from a buffer, 16 bytes a lane from byte lane_at + at of it on, and known to
// the compiler: loads ahead of it that it waits for do not wait for the copies. (As
// global_load_lds a copy may be one of LDS to the compiler's counts, and it then waits
// for all that is in flight.)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t weight_rows(const void* from,
                                                              int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(from), 0, bytes,
                                           0x00020000);
}
__device__ __forceinline__ void copy_rows_to_lds(__amdgpu_buffer_rsrc_t from,
                                                 int lane_at, int at,
                                                 char* base) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      from, (__attribute__((address_space(3))) void*)base, 16, lane_at, at, 0,
      0);
}

// 16 bytes at any address
typedef __attribute__((ext_vector_type(4), aligned(1))) int i32x4_any;

// The same copy of 16 bytes a lane where the sources need not start at their
// multiples, as that asks: through a register, and waited for.
template <bool ALIGNED>
__device__ __forceinline__ void to_lds(const void* src, char* base) {
  if constexpr (ALIGNED)
    copy_to_lds(src, base);
  else
    *reinterpret_cast<i32x4*>(base + (threadIdx.x & 63) * 16) =
        *reinterpret_cast<const i32x4_any*>(src);
}

// Workgroups go round the eight XCDs one by one: number b of n such that
// each XCD (an L2 cache of its own) gets a contiguous run of numbers.
__device__ __forceinline__ int xcd_run(int b, int n) {
  const int per = n / 8, rem = n % 8, xcd = b % 8;
  return (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) +
         b / 8;
}

// The chunk of n, of 128 bytes of a row, with which workgroup b of a product of
// few rows begins; it goes round from there. Workgroups that all begin at the
// start of rows whose strides are large powers of two ask the same few memory
// channels: us, that and this, 32 rows of 32768 x 4096 59.8 and 51.4, 64 of 16384 x
// 8192 gated 65.0 and 54.0, of 28672 x 4096 gated 55.7 and 51.1, one row 45.3 and
// 42.5, of 4096 x 14336 25.6 and 23.0. STEP is the best of a dozen odd numbers in a
// form, most of them within 3%. Rows of less than 32 chunks gain nothing (151936 x
// 1536 115.0, 114.3) and are spared the division (24 rows of 768 x 768 3.24, 3.33).
template <int STEP>
__device__ __forceinline__ int chunk_turn(int b, int n) {
  return n < 32 ? 0 : (int)((unsigned)(b * STEP) % (unsigned)n);
}

// Block-level reduce across NW waves using LDS scratch (NW <= 16).
template <int NW>
__device__ __forceinline__ float block_reduce_sum(float v, float* lds_scratch) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = threadIdx.x / WAVE;
  v = wave_reduce_sum(v);
  if (lane == 0) lds_scratch[wid] = v;
  __syncthreads();
  float r = (lane < NW) ? lds_scratch[lane] : 0.f;
  r = wave_reduce_sum(r);
  // broadcast via readfirstlane semantics: all lanes of wave 0 now agree
  if (threadIdx.x == 0) lds_scratch[0] = r;
  __syncthreads();
  float out = lds_scratch[0];
  __syncthreads();
  return out;
}

#define HIP_CHECK_KERNEL()                                                    \
  do {                                                                        \
    hipError_t e = hipGetLastError();                                         \
    if (e != hipSuccess) {                                                    \
      printf("HIP kernel launch error: %s\n", hipGetErrorString(e));          \
    }                                                                         \
  } while (0)

// Branch-free transcendentals on the native v_exp_f32 / v_rcp_f32
// instructions. libm tanhf/erff/expf compile to branchy range-checked
// slow paths (one s_and_saveexec waterfall per element — measured 37%
// of a fused-GELU GEMM's time); these stay straight-line VALU.
__device__ __forceinline__ float fast_exp(float x) {
  return __builtin_amdgcn_exp2f(x * 1.4426950408889634f);
}
__device__ __forceinline__ float fast_rcp(float x) {
  return __builtin_amdgcn_rcpf(x);  // ~1 ulp: plenty for bf16 outputs
}
__device__ __forceinline__ float fast_tanh(float u) {
  // 1 - 2/(e^{2u}+1); exp2 under/overflow saturates to +-1 gracefully
  const float e = __builtin_amdgcn_exp2f(u * 2.885390081777927f);
  return 1.f - 2.f * fast_rcp(e + 1.f);
}
__device__ __forceinline__ float fast_erf(float z) {
  // Abramowitz-Stegun 7.1.26 (max abs err 1.5e-7), branch-free
  const float a = fabsf(z);
  const float t = fast_rcp(fmaf(0.3275911f, a, 1.f));
  float p = fmaf(1.061405429f, t, -1.453152027f);
  p = fmaf(p, t, 1.421413741f);
  p = fmaf(p, t, -0.284496736f);
  p = fmaf(p, t, 0.254829592f);
  const float y = 1.f - p * t * fast_exp(-a * a);
  return copysignf(y, z);
}
__device__ __forceinline__ float fast_gelu(float x) {
  // tanh approximation (matches BERT/HF "gelu_new" semantics)
  const float k0 = 0.7978845608028654f;  // sqrt(2/pi)
  const float k1 = 0.044715f;
  return 0.5f * x * (1.f + fast_tanh(k0 * (x + k1 * x * x * x)));
}
// the same on library functions
__device__ __forceinline__ float gelu_exact(float x) {
  return 0.5f * x *
         (1.f + tanhf(0.7978845608028654f * (x + 0.044715f * x * x * x)));
}
__device__ __forceinline__ float gelu_erf(float x) {
  return 0.5f * x * (1.f + fast_erf(x * 0.70710678118654752f));
}
__device__ __forceinline__ float silu(float x) {
  return x * fast_rcp(1.f + fast_exp(-x));
}
// Clamped gated unit (see clamped_glu.hip): the fast form for 16-bit
// outputs and the form on library functions for 32-bit ones.
__device__ __forceinline__ float clamped_glu(float gate, float up,
                                             float limit, float alpha,
                                             float shift) {
  const float g = fminf(gate, limit);
  const float u = fminf(fmaxf(up, -limit), limit);
  return g * fast_rcp(1.f + fast_exp(-alpha * g)) * (u + shift);
}
__device__ __forceinline__ float clamped_glu_exact(float gate, float up,
                                                   float limit, float alpha,
                                                   float shift) {
  const float g = fminf(gate, limit);
  const float u = fminf(fmaxf(up, -limit), limit);
  return g / (1.f + expf(-alpha * g)) * (u + shift);
}

// xIELU with ap = softplus(p), an = softplus(q): the fast form for 16-bit
// outputs and the form on library functions for 32-bit ones.
__device__ __forceinline__ float softplus_exact(float z) {
  return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z)));
}
__device__ __forceinline__ float xielu(float z, float ap, float an) {
  const float neg = (0.5f + an) * (fast_exp(fminf(z, 0.f)) - 1.f - z);
  return 0.5f * z + (z > 0.f ? ap * z * z : neg);
}
__device__ __forceinline__ float xielu_exact(float z, float ap, float an) {
  const float neg = (0.5f + an) * (expm1f(fminf(z, 0.f)) - z);
  return 0.5f * z + (z > 0.f ? ap * z * z : neg);
}
__device__ __forceinline__ float relu2(float z) {
  const float r = fmaxf(z, 0.f);
  return r * r;
}
__device__ __forceinline__ float sigmoid_exact(float z) {
  return 1.f / (1.f + expf(-z));
}

// Scalars of the two tensor types as fp32.
__device__ __forceinline__ float to_f(unsigned short v) { return bf2f(v); }
__device__ __forceinline__ float to_f(float v) { return v; }
__device__ __forceinline__ void from_f(unsigned short* p, float v) {
  *p = f2bf(v);
}
__device__ __forceinline__ void from_f(float* p, float v) { *p = v; }

// Eight consecutive numbers of a bf16 or fp32 array, as fp32.
template <typename T>
__device__ __forceinline__ void load8(const T* p, float* f);
template <>
__device__ __forceinline__ void load8<unsigned short>(const unsigned short* p,
                                                      float* f) {
  bf8_to_f32(*reinterpret_cast<const s16x8*>(p), f);
}
template <>
__device__ __forceinline__ void load8<float>(const float* p, float* f) {
  const f32x4 a = *reinterpret_cast<const f32x4*>(p);
  const f32x4 b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[i] = a[i];
    f[4 + i] = b[i];
  }
}
__device__ __forceinline__ void store8(unsigned short* p, const float* f) {
  s16x8 v;
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = (short)f2bf(f[i]);
  *reinterpret_cast<s16x8*>(p) = v;
}
__device__ __forceinline__ void store8(float* p, const float* f) {
  f32x4 a, b;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    a[i] = f[i];
    b[i] = f[4 + i];
  }
  *reinterpret_cast<f32x4*>(p) = a;
  *reinterpret_cast<f32x4*>(p + 4) = b;
}
