// Inner products of queries with the rows of a corpus, float32 in and out:
// S[q, n] = sum_k Q[q, k] C[n, k].
//
// The card's float32 products reach 136 TFLOP/s here; its bf16 products are
// ten times as fast. A float32 number is the sum of three bf16 numbers of 8
// bits each, exactly (hi, mid, lo: what rounding leaves is representable), so
// six bf16 products, hi hi, hi mid, mid hi, mid mid, hi lo, lo hi, accumulated
// in float32, leave out what is below 2^-24 of a product. The first has sums
// of its own, so that the running sum is rounded once in 32 products.
//
// A workgroup of 8 waves has QT queries and 128 rows of the corpus, in steps
// of 32 columns. Queries are split once ahead (split_kernel) and go to LDS as
// they lie; rows of the corpus pass through registers, where they are split:
// once each for up to 256 queries. Two buffers, one barrier a step; the next
// step's copies and rows are in flight behind the products of this one, and
// there when the rows are split (the wait for the rows is one for the younger
// copies too). A wave has QT / 4 queries by 64 rows: the 24 fragments of a step
// feed 96 products, which bound it.
// Where a sum comes out infinite or NaN (numbers of the operands that are, or
// that exceed bf16), it is done again in plain float32.
//
// Measured at 250000 rows of 768, us, library product and this: 64 queries 214
// -> 185, 128 404 -> 279, 256 716 -> 487 (1.2 PFLOP/s of bf16 products; below
// 64 the reading of the corpus bounds both). Error against 64 bits of unit
// vectors, rms and largest: 1.8e-8 -> 5.8e-9 and 2.6e-7 -> 7.4e-8.
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

extern __shared__ __attribute__((aligned(16))) char smem[];

#define SC_CT 128  // rows of the corpus
#define SC_BK 32

__device__ __forceinline__ unsigned int sc_pack(float a, float b) {
  return __builtin_bit_cast(
      unsigned int, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
__device__ __forceinline__ float sc_lo(unsigned int v) {
  return __builtin_bit_cast(float, v << 16);
}
__device__ __forceinline__ float sc_hi(unsigned int v) {
  return __builtin_bit_cast(float, v & 0xffff0000u);
}
// four numbers as three times four bf16
__device__ __forceinline__ void sc_split(f32x4 x, i32x2 (&out)[3]) {
#pragma unroll
  for (int p = 0; p < 3; ++p)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const unsigned int v = sc_pack(x[2 * i], x[2 * i + 1]);
      out[p][i] = (int)v;
      x[2 * i] -= sc_lo(v);
      x[2 * i + 1] -= sc_hi(v);
    }
}

// place of piece c (of 16 bytes, 4 a row) of row r in a plane of 64-byte rows
__device__ __forceinline__ int sc_at(int r, int c) {
  return r * 64 + ((c ^ (r >> 1 & 3)) * 16);
}

// Queries [Q, K] as planes by step: [K / 32][tiles][3][QT rows of 64 bytes],
// laid out as in LDS; rows past Q are 0.
__global__ void __launch_bounds__(256)
score_split_kernel(const float* __restrict__ q, char* __restrict__ planes,
                   int Q, int K, int QT, int tiles) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;  // four columns each
  const int per = K / 4;
  const int row = (int)(i / per), c = (int)(i % per) * 4;
  if (row >= tiles * QT) return;
  f32x4 x = {0.f, 0.f, 0.f, 0.f};
  if (row < Q) x = *reinterpret_cast<const f32x4*>(q + (long)row * K + c);
  i32x2 s[3];
  sc_split(x, s);
  const int r = row % QT;
  char* dst = planes +
              ((long)(c / SC_BK) * tiles + row / QT) * (3 * QT * 64) +
              sc_at(r, c % SC_BK / 8) + (c & 4) * 2;
#pragma unroll
  for (int p = 0; p < 3; ++p)
    *reinterpret_cast<i32x2*>(dst + p * QT * 64) = s[p];
}

// corpus is not __restrict__: its loads are counted by the waits in the loop,
// together with the copies in assembly, so they must stay in their place among
// those. Memory that assembly may write orders them; memory that nothing else
// reaches would not.
template <int QT>
__global__ void __launch_bounds__(512, 2)
score_kernel(const float* __restrict__ q, const char* __restrict__ planes,
             const float* corpus, float* __restrict__ out, int Q, int N,
             int K, int tiles) {
  constexpr int MI = QT / 64;            // query blocks of a wave
  constexpr int QB = 3 * QT * 64;        // bytes of the queries of a step
  constexpr int BUF = QB + 3 * SC_CT * 64;
  constexpr int COPIES = QB / 1024;      // of 1 KiB
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i16 = lane & 15, g = lane >> 4;
  const int qw = wid & 3, cw = wid >> 2;
  const int bid = xcd_run(blockIdx.x, gridDim.x);
  const int tq = bid % tiles, tc = bid / tiles;
  const int nk = K / SC_BK;

  // corpus rows threadIdx / 8 and 64 on, 16 bytes each
  const int cr = threadIdx.x >> 3, cc = threadIdx.x & 7;
  const float* src[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
    src[i] = corpus + (long)min(tc * SC_CT + i * 64 + cr, N - 1) * K + cc * 4;
  f32x4 reg[2];
  auto load = [&](int k) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      reg[i] = *reinterpret_cast<const f32x4*>(src[i] + k * SC_BK);
  };
  auto store = [&](char* buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      i32x2 s[3];
      sc_split(reg[i], s);
      char* dst = buf + QB + sc_at(i * 64 + cr, cc >> 1) + (cc & 1) * 8;
#pragma unroll
      for (int p = 0; p < 3; ++p)
        *reinterpret_cast<i32x2*>(dst + p * SC_CT * 64) = s[p];
    }
  };
  auto copy = [&](int k, char* buf) {
    const char* from = planes + ((long)k * tiles + tq) * QB + lane * 16;
#pragma unroll
    for (int i = 0; i < (COPIES + 7) / 8; ++i)
      if (COPIES % 8 == 0 || i * 8 + wid < COPIES)
        copy_to_lds(from + (i * 8 + wid) * 1024, buf + (i * 8 + wid) * 1024);
  };

  f32x4 acc[4][MI], low[4][MI];  // of hi hi, of the rest
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < MI; ++j)
      acc[i][j] = low[i][j] = {0.f, 0.f, 0.f, 0.f};

  copy(0, smem);
  load(0);
  store(smem);
  if (nk > 1) load(1);
  for (int k = 0; k < nk; ++k) {
    char* buf = smem + (k & 1) * BUF;
    // this step's copies (the two loads of the next corpus rows came after
    // them), its split rows, the reads of the other buffer
    if (k + 1 < nk)
      asm volatile("s_waitcnt vmcnt(2) lgkmcnt(0)" ::: "memory");
    else
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (k + 1 < nk) copy(k + 1, smem + (~k & 1) * BUF);
    bf16x8 cf[3][4], qf[3][MI];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        cf[p][i] = *reinterpret_cast<const bf16x8*>(
            buf + QB + p * SC_CT * 64 + sc_at(cw * 64 + i * 16 + i16, g));
#pragma unroll
      for (int j = 0; j < MI; ++j)
        qf[p][j] = *reinterpret_cast<const bf16x8*>(
            buf + p * QT * 64 + sc_at((qw * MI + j) * 16 + i16, g));
    }
#pragma unroll
    for (int pair = 0; pair < 6; ++pair) {
      constexpr int PC[6] = {2, 0, 1, 1, 0, 0};
      constexpr int PQ[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < MI; ++j) {
          f32x4& to = pair == 5 ? acc[i][j] : low[i][j];
          to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              cf[PC[pair]][i], qf[PQ[pair]][j], to, 0, 0, 0);
        }
    }
    if (k + 1 < nk) {
      store(smem + (~k & 1) * BUF);
      if (k + 2 < nk) load(k + 2);
    }
  }

#pragma unroll
  for (int j = 0; j < MI; ++j) {
    const int row = tq * QT + (qw * MI + j) * 16 + i16;
    if (row >= Q) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = tc * SC_CT + cw * 64 + i * 16 + g * 4;
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = acc[i][j][e] + low[i][j][e];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (!(fabsf(v[e]) < INFINITY) && n + e < N) {
          float s = 0.f;
          for (int c = 0; c < K; ++c)
            s = fmaf(q[(long)row * K + c], corpus[(long)(n + e) * K + c], s);
          v[e] = s;
        }
      float* o = out + (long)row * N + n;
      if (N % 4 == 0 && n < N)
        *reinterpret_cast<f32x4*>(o) = v;
      else
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) o[e] = v[e];
    }
  }
}

// queries of a workgroup for Q of them
extern "C" int score_tile(int Q) { return Q <= 64 ? 64 : Q <= 128 ? 128 : 256; }

extern "C" void launch_score(const float* q, void* planes,
                             const float* corpus, float* out, int Q, int N,
                             int K, hipStream_t stream) {
  const int QT = score_tile(Q), tiles = (Q + QT - 1) / QT;
  const long quads = (long)tiles * QT * (K / 4);
  hipLaunchKernelGGL(score_split_kernel, dim3((quads + 255) / 256), dim3(256),
                     0, stream, q, (char*)planes, Q, K, QT, tiles);
#define SC(T)                                                               \
  hipLaunchKernelGGL(score_kernel<T>,                                       \
                     dim3((N + SC_CT - 1) / SC_CT * tiles), dim3(512),      \
                     2 * 3 * (T + SC_CT) * 64, stream, q, (const char*)planes, \
                     corpus, out, Q, N, K, tiles)
  if (QT == 64) SC(64);
  else if (QT == 128) SC(128);
  else SC(256);
#undef SC
}
