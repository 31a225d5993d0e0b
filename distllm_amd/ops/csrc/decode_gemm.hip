// Products of few rows: out[M,N] = x[M,K] @ W[N,K]^T, M <= 256 and, of few
// columns or a short K, up to some thousand, with bias
// and activation in the same launch where K is not split over workgroups.
// Replaces the skinny-M GEMMs vLLM issues per decode step (reference
// delegated generation to vLLM, distllm/generate/generators/
// vllm_backend.py:30-68).
//
// Every weight is used by one wave once, so the weights' way from memory is
// the cost. What decides the form is what else goes through the CU's load
// path: a load whose lanes are 16 rows x 64 bytes, which is what an MFMA
// operand wants, takes it 64 cycles for 1 KiB where whole lines take 16, and
// 6 TB/s leave about 100 cycles per KiB of weights.
//
//  ring    M <= 16 but for many columns of a short K, and up to 64 where
//          columns are few. A workgroup has 16 columns (rows of W), of up to
//          2048 columns 8, and its 4 waves take the 64-wide chunks of K in turn;
//          W and x pass through a ring of LDS buffers that belongs to the wave
//          alone: whole lines by global_load_lds, counted waits, no barriers. The waves' sums meet in LDS: no slabs, no second
//          launch. (W straight to operand registers is 2% faster for one row
//          of 28672 x 4096 and up, and 10 to 60% slower else.)
//  tile    above: W and x tiles of 64 columns of K in a ring that 4 or 8
//          waves share, one barrier per chunk; where N alone does not fill
//          the chip K is split over workgroups and a second launch sums fp32
//          slabs. Some hundred rows go by blocks of 64 (mid_gemm_shares).
//  even    17 to 64 rows where tiles of 48 to 128 columns come out even on the
//          card's CUs and those of 64 do not.
//
// Measured in a graph over fresh weights, us (GB/s of weights); before: the
// faster of a two-stage tile of 128 rows with slabs and the library:
//   M = 1   28672 x 4096 gated 64 -> 41 (5.7 TB/s), 6144 x 4096 20 -> 11.3,
//           4096 x 4096 12 -> 8.1, 4096 x 14336 31 -> 23.3, 32768 x 4096 58 ->
//           45 (6.0 TB/s), 768 x 768 5.1 -> 2.7
//   M = 64  28672 x 4096 gated 57 -> 51 (as tiles; even 45 to 49), 6144 x 4096
//           25 -> 17.6, 4096 x 4096 18 -> 12.4, 4096 x 14336 38 -> 28.4, 768 x 768
//           7 -> 3.8
//
// Both LDS images hold rows of 128 bytes whose 16-byte pieces are XOR-ed
// with the row, on the source address of the copies.
#include "common.h"
#include "gelu_rows.h"
#include "norm_row.h"
#include <climits>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef unsigned short u16;

extern __shared__ __attribute__((aligned(16))) char smem[];

// what follows the sum: bias, activation, store
enum DgAct { DG_NONE = 0, DG_SWIGLU = 1, DG_CLAMPED = 2, DG_XIELU = 3,
             DG_ROWS = 4, DG_RELU2 = 5, DG_GELU_TANH = 6, DG_GELU_ERF = 7,
             DG_SILU = 8,
             DG_F32 = 9 };  // none, and the 16-bit numbers are stored as 32

struct DgEnd {
  const u16* bias;
  u16* out;
  int M, N;  // of the product; gated units have N / 2 columns of output
  float limit, alpha, shift;
  const float* nums;
  RowsArgs rows;
};

constexpr bool dg_glu(int act) { return act == DG_SWIGLU || act == DG_CLAMPED; }

// columns n .. n + 3 of row m; of a gated unit v is the gate and u the
// up-projection
template <int ACT>
__device__ __forceinline__ void dg_finish(const DgEnd& e, int m, int n,
                                          f32x4 v, f32x4 u) {
  const int cols = dg_glu(ACT) ? e.N / 2 : e.N;
  float ap = 0.f, an = 0.f;
  if (ACT == DG_XIELU) {
    ap = softplus_exact(e.nums[0]);
    an = softplus_exact(e.nums[1]);
  }
  u16 o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = v[i], b = u[i];
    if (e.bias != nullptr) {
      a += bf2f(e.bias[n + i]);
      if (dg_glu(ACT)) b += bf2f(e.bias[cols + n + i]);
    }
    if (ACT == DG_SWIGLU) a = silu(a) * b;
    if (ACT == DG_CLAMPED) a = clamped_glu(a, b, e.limit, e.alpha, e.shift);
    if (ACT == DG_XIELU) a = xielu(a, ap, an);
    if (ACT == DG_ROWS)
      a = n + i < e.rows.n
              ? fast_gelu(a) *
                    bf2f(((const u16*)e.rows.table)[e.rows.tokens[m] *
                                                        e.rows.ld +
                                                    e.rows.col0 + n + i])
              : 0.f;
    if (ACT == DG_RELU2) a = relu2(a);
    if (ACT == DG_GELU_TANH) a = fast_gelu(a);
    if (ACT == DG_GELU_ERF) a = gelu_erf(a);
    if (ACT == DG_SILU) a = silu(a);
    o[i] = f2bf(a);
  }
  if constexpr (ACT == DG_F32)
    *reinterpret_cast<f32x4*>((float*)(void*)e.out + (long)m * cols + n) =
        f32x4{bf2f(o[0]), bf2f(o[1]), bf2f(o[2]), bf2f(o[3])};
  else
    *reinterpret_cast<i32x2*>(e.out + (long)m * cols + n) =
        *reinterpret_cast<const i32x2*>(o);
}

__device__ __forceinline__ void dg_copy(const u16* src, char* dst) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) unsigned int*)src,
      (__attribute__((address_space(3))) unsigned int*)dst, 16, 0, 0);
}
template <int N>
__device__ __forceinline__ void dg_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}

// rows of W of a workgroup's column block: 16 at a time, of a gated unit
// gate rows and up rows in turn
template <bool GLU>
__device__ __forceinline__ int dg_wrow(int block0, int t16, int N) {
  if (GLU) return block0 + (t16 >> 1) * 16 + (t16 & 1) * (N / 2);
  return block0 + t16 * 16;
}

// The sums of the NW waves that share K, added up: 16 x 16 tiles in LDS,
// [wave][NT][MT], of which this wave has COUNT from `first` on.
template <int ACT, int MT, int NT, int NW, int COUNT = 1, bool HALF = false>
__device__ __forceinline__ void dg_join(const DgEnd& e, int n0, int first,
                                        const f32x4* acc) {
  constexpr bool GLU = dg_glu(ACT);
  const int lane = threadIdx.x & 63;
  float* red = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int i = 0; i < COUNT; ++i)
    *reinterpret_cast<f32x4*>(red + (first + i) * 256 + lane * 4) = acc[i];
  __syncthreads();
  constexpr int UNITS = (GLU ? NT / 2 : NT) * MT * 64;
  for (int k = threadIdx.x; k < UNITS; k += blockDim.x) {
    const int l = k & 63, tj = (k >> 6) % MT, ti = (k >> 6) / MT;
    const int m = tj * 16 + (l & 15);
    if (m >= e.M || (HALF && l >= 32)) continue;
    f32x4 v = {0.f, 0.f, 0.f, 0.f}, u = v;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float* p =
          red + ((w * NT + ti * (GLU ? 2 : 1)) * MT + tj) * 256 + l * 4;
      v += *reinterpret_cast<const f32x4*>(p);
      if (GLU) u += *reinterpret_cast<const f32x4*>(p + MT * 256);
    }
    dg_finish<ACT>(e, m, n0 + ti * 16 + (l >> 4) * 4, v, u);
  }
}

// ---- ring -------------------------------------------------------------------
constexpr int dg_ring_lds(int MT, int NT, int NW, int R) {
  const int ring = NW * R * (NT + MT) * 2048, sums = NW * NT * MT * 1024;
  return ring > sums ? ring : sums;
}

// XP: eights of rows of x, as many as M has; what lies in LDS in the place of
// others of the MT sixteens makes no result that is kept. Of few columns the copies
// are the cost, most of them x's. us in a graph over fresh weights, all rows of 16, 32
// or 64 copied and those that are: 768 x 3072, 1 row 4.12 and 4.00, 24 5.03 and 4.87,
// 40 6.98 and 6.04, 48 7.03 and 6.46; 2304 x 768, 24 3.31 and 3.30, 40 3.85 and 3.56;
// 2048 x 2048, 1 4.37 and 4.24, 40 6.90 and 6.49; 4096 x 14336, 1 23.3 and 23.1.
// HALF: 8 columns a workgroup, where those of all still fit the card at once. Half of
// the matrix cores' rows are for nothing, but a CU takes in less: us as above, 16 and 8
// columns, 1, 8, 24, 64 rows: 768 x 3072 4.6, 5.1, 6.6, 10.1 and 4.5, 4.6, 5.8, 9.4; 768
// x 768 2.7, 2.8, 3.1, 3.9 and 2.7, 2.8, 3.0, 3.8; 1024 x 4096 5.5, 6.0, 7.9, 12.1 and
// 5.3, 5.4, 6.9, 11.3; 2048 x 2048 4.3, 4.6, 5.5, 7.7 and 4.1, 4.2, 5.0, 7.4; in two
// rounds, 2304 x 768, 2.8, 2.9, 3.2, 4.0 and 2.9, 3.0, 4.6, 6.1.
template <int ACT, int XP, int NT, int NW, int R, bool HALF = false>
__global__ void __launch_bounds__(NW * 64)
dg_ring_kernel(const u16* __restrict__ X, const u16* __restrict__ W, int K,
               const DgEnd e) {
  constexpr bool GLU = dg_glu(ACT);
  constexpr int MT = (XP + 1) / 2;
  constexpr int WP = HALF ? 1 : 2;  // eights of rows of W
  static_assert(!HALF || (NT == 1 && !GLU), "one half of 16 columns");
  constexpr int STAGE = (NT + MT) * 2048, LOADS = NT * WP + XP;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * (GLU || HALF ? NT * 8 : NT * 16);
  char* ring = smem + wid * R * STAGE;
  const int lr = lane >> 3, lc = ((lane & 7) ^ lr) * 8;
  const u16* src[NT + MT][2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
      src[t][p] = W + (long)(dg_wrow<GLU>(n0, t, e.N) + p * 8 + lr) * K + lc;
#pragma unroll
    for (int t = 0; t < MT; ++t)
      src[NT + t][p] =
          X + (long)min(t * 16 + p * 8 + lr, e.M - 1) * K + lc;
  }
  // chunks wid, wid + NW, ... from the block's first one on: halves have that of the
  // 16 columns, so that a column's sum has one order in all forms (it costs nothing)
  const int nch = K / 64, mine = (nch - wid + NW - 1) / NW;
  const int turn =
      chunk_turn<37>(HALF ? blockIdx.x / 2 : blockIdx.x, nch) + wid;
  auto issue = [&](int c) {
    char* dst = ring + (c % R) * STAGE + lane * 16;
    int k = c * NW + turn;
    if (k >= nch) k -= nch;
#pragma unroll
    for (int t = 0; t < NT + MT; ++t)
#pragma unroll
      for (int p = 0; p < 2; ++p)
        if (t < NT ? p < WP : (t - NT) * 2 + p < XP)
          dg_copy(src[t][p] + (long)k * 64, dst + t * 2048 + p * 1024);
  };
  f32x4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = {0.f, 0.f, 0.f, 0.f};
  auto compute = [&](int c) {
    const char* b = ring + (c % R) * STAGE;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      bf16x8 f[NT + MT];
#pragma unroll
      for (int t = 0; t < NT + MT; ++t)
        f[t] = *reinterpret_cast<const bf16x8*>(
            b + t * 2048 + r * 128 + (((h * 4 + g) ^ (r & 7)) * 16));
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              f[i], f[NT + j], acc[i][j], 0, 0, 0);
    }
    // the buffer is read before the wave fills it again
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  if (mine >= R - 1) {
    for (int c = 0; c < R - 1; ++c) issue(c);
    int c = 0;
    for (; c + R - 1 < mine; ++c) {
      issue(c + R - 1);
      dg_wait<(R - 1) * LOADS>();
      compute(c);
    }
    static_assert(R == 3 || R == 4, "tail");
    if constexpr (R == 4) {
      dg_wait<2 * LOADS>();
      compute(c++);
    }
    dg_wait<LOADS>();
    compute(c++);
    dg_wait<0>();
    compute(c);
  } else {
    for (int c = 0; c < mine; ++c) issue(c);
    dg_wait<0>();
    for (int c = 0; c < mine; ++c) compute(c);
  }
  __syncthreads();
  dg_join<ACT, MT, NT, NW, NT * MT, HALF>(e, n0, wid * NT * MT, &acc[0][0]);
}

// ---- ring with the norm ahead of the product --------------------------------
// One row (norm_row.h). The normed row stays in LDS, so that the rings hold
// weights only: more of them. Measured in a graph, us, norm and product in two
// launches and in one: 28672 x 4096 gated 45.8 and 41.3, 6144 x 4096 14.3 and
// 11.8, 4096 x 2048 7.4 and 5.8 (the weights as copies that the compiler counts one
// by one, so that the norm does not wait for them); two rows normed by every workgroup 46.5 and
// 49.1 at the first.
constexpr int dg_norm_lds(int K, int NT, int R) {
  return 128 + K * 2 + 4 * R * NT * 2048;
}
// chunks that every wave has at least: R - 1 are started ahead of the norm
constexpr int dg_norm_ring(int NT) { return NT == 2 ? 4 : 6; }

template <int ACT, int NT, int NC>
__global__ void __launch_bounds__(256)
dg_norm_ring_kernel(const NormRow n, const u16* __restrict__ W, int K,
                    const DgEnd e) {
  constexpr bool GLU = dg_glu(ACT);
  constexpr int NW = 4, R = dg_norm_ring(NT);
  constexpr int STAGE = NT * 2048, LOADS = NT * 2;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * (GLU ? NT * 8 : NT * 16);
  char* hs = smem + 128;
  char* ring = hs + K * 2 + wid * R * STAGE;
  const int lr = lane >> 3;
  const int lane_at = lr * K * 2 + ((lane & 7) ^ lr) * 16;
  __amdgpu_buffer_rsrc_t src[NT];  // 16 rows of W
#pragma unroll
  for (int t = 0; t < NT; ++t)
    src[t] = weight_rows(W + (long)dg_wrow<GLU>(n0, t, e.N) * K, 32 * K);
  // chunks wid, wid + NW, ... from the block's first one on
  const int nch = K / 64, mine = (nch - wid + NW - 1) / NW;
  const int turn = chunk_turn<37>(blockIdx.x, nch) + wid;
  auto chunk = [&](int c) {
    const int k = c * NW + turn;
    return k >= nch ? k - nch : k;
  };
  auto issue = [&](int c) {
    char* dst = ring + (c % R) * STAGE;
    const int k = chunk(c) * 128;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int p = 0; p < 2; ++p)
        copy_rows_to_lds(src[t], lane_at, k + p * 16 * K,
                         dst + t * 2048 + p * 1024);
  };
  norm_row<NC>(n, K, reinterpret_cast<float*>(smem), hs, [&]() {
#pragma unroll
    for (int c = 0; c < R - 1; ++c) issue(c);
  });

  f32x4 acc[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) acc[i] = {0.f, 0.f, 0.f, 0.f};
  auto compute = [&](int c) {
    const char* b = ring + (c % R) * STAGE;
    const char* xs = hs + chunk(c) * 128;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bf16x8 x =
          *reinterpret_cast<const bf16x8*>(xs + (h * 4 + g) * 16);
#pragma unroll
      for (int i = 0; i < NT; ++i)
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            *reinterpret_cast<const bf16x8*>(
                b + i * 2048 + r * 128 + (((h * 4 + g) ^ (r & 7)) * 16)),
            x, acc[i], 0, 0, 0);
    }
    // the buffer is read before the wave fills it again
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  int c = 0;
  for (; c + R - 1 < mine; ++c) {
    issue(c + R - 1);
    dg_wait<(R - 1) * LOADS>();
    compute(c);
  }
  dg_wait<0>();
  for (; c < mine; ++c) compute(c);
  __syncthreads();
  dg_join<ACT, 1, NT, NW, NT>(e, n0, wid * NT, acc);
}

template <int ACT>
static void dg_norm_launch(const NormRow& n, const u16* W, int K,
                           const DgEnd& e, hipStream_t st) {
  constexpr int NT = dg_glu(ACT) ? 2 : 1;
#define DG_NR(NC)                                                          \
  hipLaunchKernelGGL((dg_norm_ring_kernel<ACT, NT, NC>),                   \
                     dim3(e.N / (NT * 16)), dim3(256),                     \
                     dg_norm_lds(K, NT, dg_norm_ring(NT)), st, n, W, K, e)
  if (K <= 2048) DG_NR(1);
  else if (K <= 4096) DG_NR(2);
  else DG_NR(4);  // up to 8192
#undef DG_NR
}

// act 0, 1 or 9: product (of 16 or 32 bits) or gated unit (SwiGLU) of the norm of
// one row. K from
// 1280 (five chunks of 64 for each of four waves) to 8192.
extern "C" void launch_norm_gemm(const void* a, const void* b,
                                 const void* w_norm, void* sum, float eps,
                                 const void* W, const void* bias, void* out,
                                 int N, int K, int act, hipStream_t stream) {
  const NormRow n = {(const u16*)a, (const u16*)b, (const u16*)w_norm,
                     (u16*)sum, eps};
  const DgEnd e = {(const u16*)bias, (u16*)out, 1, N, 0.f, 0.f, 0.f, nullptr,
                   {}};
  if (act == 1) dg_norm_launch<DG_SWIGLU>(n, (const u16*)W, K, e, stream);
  else if (act == 9) dg_norm_launch<DG_F32>(n, (const u16*)W, K, e, stream);
  else dg_norm_launch<DG_NONE>(n, (const u16*)W, K, e, stream);
}

// ---- tile -------------------------------------------------------------------
// MP rows of x, 64 of W. Waves: 4 for MP = 32 and 8 else, WN of them side by
// side over the columns.
constexpr int dg_tile_lds(int MP, int R) { return R * (MP + 64) * 128; }

template <int ACT, int MP, int R, bool SLAB>
__global__ void __launch_bounds__(MP == 32 ? 256 : 512)
dg_tile_kernel(const u16* __restrict__ X, const u16* __restrict__ W,
               float* __restrict__ slabs, int K, int splitk, const DgEnd e) {
  constexpr bool GLU = dg_glu(ACT);
  constexpr int NW = MP == 32 ? 4 : 8;
  constexpr int STAGE = (MP + 64) * 128, LOADS = STAGE / 1024 / NW;
  static_assert(LOADS * NW * 1024 == STAGE, "whole pieces per wave");
  constexpr int WN = MP <= 64 ? 2 : 1, WM = NW / WN;
  constexpr int FM = MP / 16 / WM, FN = 4 / WN;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int ncb = e.N / 64;
  const int cb = blockIdx.x % ncb, ks = blockIdx.x / ncb % splitk;
  const int m0 = blockIdx.x / ncb / splitk * MP;  // the tile's first row
  const int nt = K / splitk / 64, n0 = cb * (GLU ? 32 : 64);
  const int lr = lane >> 3, lc = ((lane & 7) ^ lr) * 8;
  const u16* src[LOADS];
#pragma unroll
  for (int p = 0; p < LOADS; ++p) {
    const int row = (wid * LOADS + p) * 8 + lr;
    src[p] = (row < 64
                  ? W + (long)(dg_wrow<GLU>(n0, row >> 4, e.N) + (row & 15)) * K
                  : X + (long)min(m0 + row - 64, e.M - 1) * K) +
             ks * (K / splitk) + lc;
  }
  // with more than 64 rows in a tile it is x that all read, and do so together: us
  // from the first columns on and from different ones, 120 rows of 4096 x 14336 41.3
  // and 48.9, 100 rows 39.9 and 42.2. Not so in blocks of 64 of more rows: 128 rows
  // of 2048 x 8192 18.2 and 17.3, 66 rows 17.1 and 16.6, 128 of 4096 x 4096 17.2 and
  // 16.8, 160 of 2048 x 4096 15.2 and 15.2
  const int turn = MP <= 64 ? chunk_turn<19>(cb, nt) : 0;
  auto issue = [&](int c) {
    char* dst = smem + (c % R) * STAGE + wid * LOADS * 1024 + lane * 16;
    const int k = c + turn < nt ? c + turn : c + turn - nt;
#pragma unroll
    for (int p = 0; p < LOADS; ++p)
      dg_copy(src[p] + (long)k * 64, dst + p * 1024);
  };
  const int wn = wid % WN, wm = wid / WN;
  f32x4 acc[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) acc[i][j] = {0.f, 0.f, 0.f, 0.f};
  auto compute = [&](int c) {
    const char* b = smem + (c % R) * STAGE;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int piece = ((h * 4 + g) ^ (r & 7)) * 16;
      bf16x8 a[FN], x[FM];
#pragma unroll
      for (int i = 0; i < FN; ++i)
        a[i] = *reinterpret_cast<const bf16x8*>(
            b + ((wn * FN + i) * 16 + r) * 128 + piece);
#pragma unroll
      for (int j = 0; j < FM; ++j)
        x[j] = *reinterpret_cast<const bf16x8*>(
            b + (64 + (wm * FM + j) * 16 + r) * 128 + piece);
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a[i], x[j], acc[i][j], 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  // a chunk's buffer is filled again after the barrier of the next chunk,
  // by when every wave has read it
  auto arrive = [&]() {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  if (nt >= R - 1) {
    for (int c = 0; c < R - 1; ++c) issue(c);
    int c = 0;
    for (; c + R - 1 < nt; ++c) {
      dg_wait<(R - 2) * LOADS>();
      arrive();
      issue(c + R - 1);
      compute(c);
    }
#pragma unroll
    for (int left = R - 2; left >= 0; --left) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"i"(left * LOADS) : "memory");
      arrive();
      compute(c++);
    }
  } else {
    for (int c = 0; c < nt; ++c) issue(c);
    dg_wait<0>();
    arrive();
    for (int c = 0; c < nt; ++c) compute(c);
  }
#pragma unroll
  for (int j = 0; j < FM; ++j) {
    const int m = m0 + (wm * FM + j) * 16 + r;
    if (m >= e.M) continue;
    if constexpr (SLAB) {
#pragma unroll
      for (int i = 0; i < FN; ++i)
        *reinterpret_cast<f32x4*>(
            slabs + ((long)ks * e.M + m) * e.N +
            dg_wrow<GLU>(n0, wn * FN + i, e.N) + g * 4) = acc[i][j];
    } else {
#pragma unroll
      for (int i = 0; i < FN; i += GLU ? 2 : 1)
        dg_finish<ACT>(e, m,
                       dg_wrow<GLU>(n0, wn * FN + i, e.N) + g * 4, acc[i][j],
                       acc[GLU ? i + 1 : i][j]);
    }
  }
}

// ---- even -------------------------------------------------------------------
// 17 to 64 rows (MP = 32 or 64 of them) by C sixteens of columns a workgroup, so many
// that the columns, or their shares of K, come out even on the card's 256 CUs. Tiles
// of 64 columns leave CUs with one or two of them beside each other (28672 columns
// are 448 tiles), and every one reads all of x again: with 112 columns that is half as
// much. One workgroup a CU, whose ring has all of LDS; 4 or 8 waves, 16 rows and half
// of the columns each. A gated unit's sixteen rows of W are eight columns of either
// kind, dealt so that a lane has both of a column.
// us in a graph over fresh weights, 64 x 64 tiles and these, 17, 32, 64 rows: 28672 x
// 4096 gated 42.7, 44.7, 49.8 and 43.7, 43.6, 45.1; 22016 x 4096 gated 39.9, 40.1, 45.3
// and 37.3, 35.8, 38.7; 27648 x 5120 gated 57.2, 60.5, 68.2 and 54.6, 53.7, 57.1; 32768
// x 4096 53.0, 52.6, 55.1 and 51.2, 50.7, 51.8; with shares of K (without what joins
// them) 6144 x 4096, 2 and 4 13.2, 12.7, 14.7 and 11.2, 11.6, 13.6; 5120 x 5120, 2 and
// 4 16.7, 18.0, 18.0 and 12.9, 12.8, 15.4.
constexpr int dg_even_stages(int MP, int C) {
  const int r = 160 * 1024 / ((C * 16 + MP) * 128);
  return r > 8 ? 8 : r;
}
constexpr int dg_even_lds(int MP, int C) {
  return dg_even_stages(MP, C) * (C * 16 + MP) * 128;
}

template <int ACT, int MP, int C, bool SLAB>
__global__ void __launch_bounds__(MP * 8)
dg_even_kernel(const u16* __restrict__ X, const u16* __restrict__ W,
               float* __restrict__ slabs, int K, int splitk, int G,
               const DgEnd e) {
  constexpr bool GLU = dg_glu(ACT);
  constexpr int NW = MP / 8, WM = MP / 16, CH = (C + 1) / 2;
  constexpr int R = dg_even_stages(MP, C), STAGE = (C * 16 + MP) * 128;
  constexpr int PIECES = STAGE / 1024, LOADS = (PIECES + NW - 1) / NW;
  static_assert((R - 1) * LOADS < 64, "copies that vmcnt counts");
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int cb = blockIdx.x % G, ks = blockIdx.x / G;
  const int F = e.N / 16;
  const int f0 = (int)((long)F * cb / G), mine = (int)((long)F * (cb + 1) / G) - f0;
  const int nt = K / splitk / 64;
  const int lr = lane >> 3, lc = ((lane & 7) ^ lr) * 8;
  const u16* src[LOADS];
  int to[LOADS];
#pragma unroll
  for (int p = 0; p < LOADS; ++p) {
    // (of uneven numbers some pieces twice)
    const int piece = min(wid * LOADS + p, PIECES - 1);
    to[p] = piece * 1024;
    const int row = piece * 8 + lr;
    const u16* from;
    if (piece < C * 2) {
      const int f = f0 + min(row >> 4, mine - 1), j = row & 15;
      const int n = GLU ? (j & 2) * (e.N / 4) + f * 8 + (j >> 2) * 2 + (j & 1)
                        : f * 16 + j;
      from = W + (long)n * K;
    } else {
      from = X + (long)min(row - C * 16, e.M - 1) * K;
    }
    src[p] = from + ks * (K / splitk) + lc;
  }
  const int turn = chunk_turn<19>(cb, nt);
  auto issue = [&](int c) {
    char* dst = smem + (c % R) * STAGE + lane * 16;
    const int k = c + turn < nt ? c + turn : c + turn - nt;
#pragma unroll
    for (int p = 0; p < LOADS; ++p) dg_copy(src[p] + (long)k * 64, dst + to[p]);
  };
  const int wn = wid % 2, wm = wid / 2;
  f32x4 acc[CH];
#pragma unroll
  for (int i = 0; i < CH; ++i) acc[i] = {0.f, 0.f, 0.f, 0.f};
  auto compute = [&](int c) {
    const char* b = smem + (c % R) * STAGE;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int piece = ((h * 4 + g) ^ (r & 7)) * 16;
      const bf16x8 x = *reinterpret_cast<const bf16x8*>(
          b + (C * 16 + wm * 16 + r) * 128 + piece);
#pragma unroll
      for (int i = 0; i < CH; ++i)
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            *reinterpret_cast<const bf16x8*>(
                b + (min(wn * CH + i, C - 1) * 16 + r) * 128 + piece),
            x, acc[i], 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  auto arrive = [&]() {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  for (int c = 0; c < R - 1; ++c) issue(c);
  int c = 0;
  for (; c + R - 1 < nt; ++c) {
    dg_wait<(R - 2) * LOADS>();
    arrive();
    issue(c + R - 1);
    compute(c);
  }
#pragma unroll
  for (int left = R - 2; left >= 0; --left) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(left * LOADS) : "memory");
    arrive();
    compute(c++);
  }
  const int m = wm * 16 + r;
  if (m >= e.M) return;
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int t = wn * CH + i;
    if (t >= mine) continue;
    if constexpr (SLAB && GLU) {
      float* to = slabs + ((long)ks * e.M + m) * e.N + (f0 + t) * 8 + g * 2;
      *reinterpret_cast<f32x2*>(to) = f32x2{acc[i][0], acc[i][1]};
      *reinterpret_cast<f32x2*>(to + e.N / 2) = f32x2{acc[i][2], acc[i][3]};
    } else if constexpr (SLAB) {
      *reinterpret_cast<f32x4*>(slabs + ((long)ks * e.M + m) * e.N +
                                (f0 + t) * 16 + g * 4) = acc[i];
    } else if constexpr (GLU) {
      const int n = (f0 + t) * 8 + g * 2, cols = e.N / 2;
      unsigned int o = 0;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        float a = acc[i][q], b = acc[i][2 + q];
        if (e.bias != nullptr) {
          a += bf2f(e.bias[n + q]);
          b += bf2f(e.bias[cols + n + q]);
        }
        a = ACT == DG_SWIGLU ? silu(a) * b
                             : clamped_glu(a, b, e.limit, e.alpha, e.shift);
        o |= (unsigned int)f2bf(a) << (q * 16);
      }
      *reinterpret_cast<unsigned int*>(e.out + (long)m * cols + n) = o;
    } else {
      dg_finish<ACT>(e, m, (f0 + t) * 16 + g * 4, acc[i], acc[i]);
    }
  }
}

// sum of fp32 slabs [splitk, M, N], four columns a thread
template <int ACT>
__global__ void __launch_bounds__(256)
dg_reduce_kernel(const float* __restrict__ slabs, int splitk, const DgEnd e) {
  constexpr bool GLU = dg_glu(ACT);
  const int cols = GLU ? e.N / 2 : e.N;
  const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= (long)e.M * cols) return;
  const int m = (int)(i / cols), n = (int)(i % cols);
  const float* p = slabs + (long)m * e.N + n;
  f32x4 v = {0.f, 0.f, 0.f, 0.f}, u = v;
  for (int s = 0; s < splitk; ++s) {
    v += *reinterpret_cast<const f32x4*>(p + (long)s * e.M * e.N);
    if (GLU) u += *reinterpret_cast<const f32x4*>(p + (long)s * e.M * e.N + cols);
  }
  dg_finish<ACT>(e, m, n, v, u);
}

// Whether 17 to 32 or 33 to 64 rows take the ring: a workgroup of it reads
// all of x for its 16 columns and fills a CU, so columns have to fit the chip
// once and K must not be long. Measured, ring and tile, in us: 32 rows 4096 x
// 4096 10.1 and 11.2, 6144 x 4096 17.1 and 15.5, 2048 x 8192 15.4 and 12.8;
// 64 rows 4096 x 1536 7.1 and 9.7, 768 x 3072 7.4 and 8.4, 5120 x 1280 10.6
// and 10.2, 2048 x 4096 12.2 and 11.5.
static bool dg_few_columns(int rows, int N, int K) {
  return N <= 4096 && K <= 4096 &&
         (long)N * K <= (rows <= 32 ? 4096L * 4096 : 4096L * 1536);
}

// Whether up to 16 rows take the tile form: a ring's workgroup has 16 columns,
// and with many columns of a short K it has hardly begun when it ends. Measured,
// ring and tile, us, 1 to 16 rows: 16384 x 128 4 and 3, 128256 x 128 19 and 9,
// 250000 x 256 53 and 28, 151936 x 512 42 and 31, 65536 x 768 20 to 22 and 18,
// 250000 x 1024 89 to 112 and 91, 65536 x 1536 34 to 41 and 38, 151936 x 1536 73
// to 95 and 87, 151936 x 2048 103 to 115 and 116.
static bool dg_short_sums(int rows, int N, int K) {
  return N >= 16384 && K <= (rows <= 8 ? 1024 : 1536);
}

// Sixteens of columns of a workgroup in the even form where `splitk` share K, 0 where
// that is another's: 3 and 5 to 8 (4 are the tile form), of which a CU has at least
// 0.85 on average, and a sum that is long enough for them. Measured over fresh weights
// at 36 numbers of columns and 13 of K, linear and gated, 17 to 64 rows, time over that
// of the tiles and shares else taken: short sums are 0.95 to 1.25 (the ring of many
// columns fills slowly, and 64 x 64 tiles are several a CU that fill each other's
// pauses), from these lines on it is 0.73 to 1.02 (6144 x 8192 by four shares 1.03):
//   3 sixteens, up to 32 rows 1536 of K, where K is shared 512; more rows 2560
//   5, up to 32 rows 768, else 1024
//   6, up to 32 rows 768, else 1536; where K is shared 1024, by eight and more 1536
//   7, 2560 (7168 columns by four shares 0.95 to 1.23: not where K is shared)
//   8, 3072, up to 32 rows 4096 and no gated unit (32768 x 4096 0.97, gated 1.04), and
//      only if they come out even to 3% (30720 x 4096 1.07)
static int dg_even_columns(int rows, int N, int K, int splitk,
                           bool gated = false) {
  if (rows <= 16 || rows > 64 || 256 % splitk) return 0;
  const int F = N / 16, G = 256 / splitk, C = (F + G - 1) / G, sum = K / splitk;
  if (C < 3 || C == 4 || C > 8 || F < 0.85f * (G * C)) return 0;
  const bool few = rows <= 32, shared = splitk > 1;
  int least = INT_MAX;
  if (C == 3) least = !few ? 2560 : shared ? 512 : 1536;
  else if (C == 5) least = few && !shared ? 768 : 1024;
  else if (C == 6) least = shared ? (splitk <= 4 ? 1024 : 1536) : few ? 768 : 1536;
  else if (C == 7) least = shared ? INT_MAX : 2560;
  else if (!shared && F >= 0.97f * (G * C) && !(few && gated))
    least = few ? 4096 : 3072;
  return sum >= least ? C : 0;
}

// How many workgroups share K in the tile and even forms: the least that give 150 of
// them, each with at least 384 of K (48 rows, in us: 4096 x 4096 2 shares
// 15.1, 4 shares 12.0, 8 shares 13.7; 4096 x 14336 39, 26.7, 29.5; 5120 x
// 1280 9.7 and 4 shares 10.6; 16384 x 4096 none 31.3, 2 shares 34.6).
static int dg_shares(int M, int N, int K) {
  int best = 1;
  for (int s = 1; s <= 16; ++s) {
    if (K % (64 * s) != 0 || (s > 1 && K / s < 384)) continue;
    best = s;
    if (N / 64 * s >= 150) break;
  }
  // twice as many where that makes tiles of 80 columns and more come out even (those
  // of 64 may be: 64 rows of 4096 x 4096, 4 and 8 shares 9.6 and 11.0)
  const int twice = best * 2;
  if (best > 1 && N / 64 * best != 256 && M <= 64 && K % (64 * twice) == 0 &&
      dg_even_columns(M, N, K, twice) >= 5)
    return twice;
  return best;
}
extern "C" int decode_gemm_shares(int M, int N, int K) {
  return M <= 16 || (M <= 64 && dg_few_columns(M, N, K)) ? 1
                                                         : dg_shares(M, N, K);
}

// The same where what follows sums the shares as it reads them, without a launch of 4.7
// us that joins them: of 17 to 32 rows the ring is the slower form then from 2048 x 4096
// on. us in a graph over fresh weights, ring and tiles, 17 and 32 rows: 2048 x 4096 8.0,
// 9.3 and 5.8, 6.1; 4096 x 4096 9.0, 11.4 and 8.5, 8.4; 4096 x 1536 5.5, 5.6 and 5.6,
// 6.0. (With the norm that sums them 4096 x 3072, three shares, 17 rows 10.6 and 10.9,
// 24 11.7 and 11.4.)
extern "C" int decode_parts_shares(int M, int N, int K) {
  if (M > 16 && M <= 32 && (long)N * K >= 2048L * 4096) {
    const int shares = dg_shares(M, N, K);
    if (shares != 3 || M >= 24) return shares;
  }
  return decode_gemm_shares(M, N, K);
}

// Whether a product of M <= 64 rows takes the ring.
extern "C" bool decode_gemm_rings(int M, int N, int K) {
  return M <= 16 ? !dg_short_sums(M, N, K)
                 : M <= 64 && dg_few_columns(M, N, K);
}

// How many workgroups share K where 65 rows and more go by tiles of 64 x 64, 0
// where another product is to be taken. Tiles have to fit the card twice over,
// and the time, 0.28 us for 64 of K (more with more than a tile a CU) and 4.5 for the
// launch that joins shares, has to stay below what the library's product costs
// either way: on the host alone 14 to 25 us a call (this one 6), and an encoder of
// some hundred rows issues its layers slower than it runs them; in a graph, over
// weights from memory, us, library (the faster of two calls) and this: 300 rows of
// 2304 x 768 10.1 and 6.9, 768 x 768 7.8 and 6.1, 3072 x 768 with GELU 10.4 and 7.4,
// 768 x 3072 (4 shares) 10.0 and 10.9, 1280 x 5120 (2) 19.6 and 17.6; 160 rows of
// 6144 x 1024 12.7 and 9.9, of 1280 x 1280 8.4 and 8.7; 1000 rows of 1024 x 1024 11.4
// and 7.9, of 768 x 3072 16.4 and 16.1. Where it is the slower one by both: 600 rows
// of 3072 x 2048 16.8 and 19.2, 1000 of 2048 x 2048 17.3 and 19.7.
extern "C" int mid_gemm_shares(int M, int N, int K) {
  if (M <= 64 || N <= 0 || N % 64 || K % 64 || K < 128) return 0;
  const long tiles = (long)((M + 63) / 64) * (N / 64);
  if (tiles > 512) return 0;
  if (K <= 1536) return 1;
  int best = 0;
  float least = 18.5f;
  for (int s = 1; s <= 4; s *= 2) {
    if (K % (64 * s) || (s > 1 && tiles * s > 256)) continue;
    const float each = tiles > 256 ? std::max(1.5f, tiles / 256.f) : 1.f;
    const float us =
        2.5f + 0.28f * (K / 64 / s) * each + (s > 1 ? 4.5f : 0.f);
    if (us >= least) continue;
    least = us;
    best = s;
  }
  return best;
}

template <int ACT>
static void dg_reduce_launch(const float* slabs, int splitk, const DgEnd& e,
                             hipStream_t st) {
  if (splitk <= 1 || e.out == nullptr) return;
  const long four = (long)e.M * (dg_glu(ACT) ? e.N / 2 : e.N) / 4;
  hipLaunchKernelGGL(dg_reduce_kernel<ACT>, dim3((four + 255) / 256),
                     dim3(256), 0, st, slabs, splitk, e);
}

template <int ACT>
static void dg_launch(const u16* X, const u16* W, float* slabs, int K,
                      int splitk, int tile, const DgEnd& e, hipStream_t st) {
  constexpr bool GLU = dg_glu(ACT);
  constexpr int NT = GLU ? 2 : 1;
#define DG_RING(XP, R)                                                       \
  hipLaunchKernelGGL((dg_ring_kernel<ACT, XP, NT, 4, R>),                    \
                     dim3(e.N / (NT * 16)), dim3(256),                       \
                     dg_ring_lds((XP + 1) / 2, NT, 4, R), st, X, W, K, e)
  // two rows of W per stage: three stages let two workgroups share a CU
  if (!tile && splitk == 1 && decode_gemm_rings(e.M, e.N, K)) {
    if constexpr (ACT == DG_NONE)
      if (e.N <= 2048) {
#define DG_HALF(XP, R)                                                       \
  hipLaunchKernelGGL((dg_ring_kernel<ACT, XP, 1, 4, R, true>),               \
                     dim3(e.N / 8), dim3(256),                               \
                     dg_ring_lds((XP + 1) / 2, 1, 4, R), st, X, W, K, e)
        if (e.M <= 8) DG_HALF(1, 4);
        else if (e.M <= 16) DG_HALF(2, 4);
        else if (e.M <= 24) DG_HALF(3, 4);
        else if (e.M <= 32) DG_HALF(4, 4);
        else if (e.M <= 40) DG_HALF(5, 4);
        else if (e.M <= 48) DG_HALF(6, 4);
        else if (e.M <= 56) DG_HALF(7, 3);
        else DG_HALF(8, 3);
#undef DG_HALF
        return;
      }
    // (one form for 32 rows and one for 64 will do for what is seldom called)
    if constexpr (ACT == DG_NONE || ACT == DG_F32 || ACT == DG_GELU_TANH ||
                  ACT == DG_GELU_ERF) {
      if (e.M <= 8) DG_RING(1, 4);
      else if (e.M <= 16) DG_RING(2, 4);
      else if (e.M <= 24) DG_RING(3, 4);
      else if (e.M <= 32) DG_RING(4, 4);
      else if (e.M <= 40) DG_RING(5, 4);
      else if (e.M <= 48) DG_RING(6, 4);
      else if (e.M <= 56) DG_RING(7, 3);
      else DG_RING(8, 3);
    } else {
      if (e.M <= 16) DG_RING(2, GLU ? 3 : 4);
      else if (e.M <= 32) DG_RING(4, 4);
      else DG_RING(8, 3);
    }
    return;
  }
#undef DG_RING
#define DG_TILE(MP, R)                                                       \
  do {                                                                       \
    const int grid = e.N / 64 * splitk * ((e.M + MP - 1) / MP);              \
    if (splitk > 1)                                                          \
      hipLaunchKernelGGL((dg_tile_kernel<ACT, MP, R, true>), dim3(grid),     \
                         dim3(MP == 32 ? 256 : 512), dg_tile_lds(MP, R), st, \
                         X, W, slabs, K, splitk, e);                         \
    else                                                                     \
      hipLaunchKernelGGL((dg_tile_kernel<ACT, MP, R, false>), dim3(grid),    \
                         dim3(MP == 32 ? 256 : 512), dg_tile_lds(MP, R), st, \
                         X, W, slabs, K, splitk, e);                         \
  } while (0)
  if constexpr (ACT == DG_NONE || ACT == DG_F32 || GLU) {
    const int C =
        tile ? 0 : dg_even_columns(e.M, e.N, K, splitk, dg_glu(ACT));
    if (C > 0) {
#define DG_EVEN(MP, CC, SL)                                                 \
  hipLaunchKernelGGL((dg_even_kernel<ACT, MP, CC, SL>), dim3(256),          \
                     dim3(MP * 8), dg_even_lds(MP, CC), st, X, W, slabs, K, \
                     splitk, 256 / splitk, e)
#define DG_EVEN_C(CC)                        \
  case CC:                                   \
    if (splitk == 1) {                       \
      if (e.M <= 32) DG_EVEN(32, CC, false); \
      else DG_EVEN(64, CC, false);           \
    } else {                                 \
      if (e.M <= 32) DG_EVEN(32, CC, true);  \
      else DG_EVEN(64, CC, true);            \
    }                                        \
    break
      switch (C) {
        DG_EVEN_C(3); DG_EVEN_C(5); DG_EVEN_C(6); DG_EVEN_C(7); DG_EVEN_C(8);
      }
#undef DG_EVEN_C
#undef DG_EVEN
      dg_reduce_launch<ACT>(slabs, splitk, e, st);
      return;
    }
  }
  const int rows = tile > 1 ? tile : e.M;
  if (rows <= 32) DG_TILE(32, 4);
  else if (rows <= 64) DG_TILE(64, 4);
  else if (rows <= 128) DG_TILE(128, 3);
  else DG_TILE(256, 3);
#undef DG_TILE
  dg_reduce_launch<ACT>(slabs, splitk, e, st);
}

// tile: the tile form whatever M is; splitk workgroups share K there. 64: by
// blocks of 64 rows. Without
// an out the slabs are left for the next kernel to sum.
extern "C" void launch_decode_gemm(const void* X, const void* W,
                                   const void* bias, void* out, void* slabs,
                                   int M, int N, int K, int splitk, int tile,
                                   int act, float limit, float alpha,
                                   float shift, const float* act_nums,
                                   const RowsArgs* rows,
                                   hipStream_t stream) {
  DgEnd e = {(const u16*)bias, (u16*)out, M, N, limit, alpha, shift, act_nums,
             {}};
  if (rows != nullptr) e.rows = *rows;
#define DG(A)                                                              \
  case A:                                                                  \
    dg_launch<A>((const u16*)X, (const u16*)W, (float*)slabs, K, splitk,   \
                 tile, e, stream);                                         \
    break
  switch (act) {
    DG(0); DG(1); DG(2); DG(3); DG(4); DG(5); DG(6); DG(7); DG(8); DG(9);
  }
#undef DG
}
