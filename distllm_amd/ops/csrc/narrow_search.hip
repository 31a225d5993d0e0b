// The best rows of a corpus for each query, float32 in and out, by way of a second
// form of the corpus of half the bytes: its numbers times a power of two as f16,
// [N, KP] (columns behind K are 0). Reading the corpus is the cost of a search of a
// few queries, and three products of f16 parts that of a batch (score.hip); one
// product of f16 numbers tells which rows can be among the best, and only these are
// scored in float32.
//
// What is left out is certain. With q' and c' the f16 forms, |q c - q' c'| is at most
// |q| |c - c'| + |q - q'| |c'| (norms) and what the sums lose, which (K + 64) 2^-23
// |q'| |c'| is more than. narrow_rows_kernel measures the largest |c - c'| and |c'| of
// a corpus, narrow_query |q - q'|, and twice the bound is the query's margin:
// k rows have products within half of it below the k-th largest one, so a row whose
// product is more than the whole below that is not among the k best. Where more than
// NS_CAP groups of four rows are within it (rows that are nearly the same), or a
// query's numbers are infinite or NaN or all 0, the query's indices say NS_UNSURE. The
// former are answered by launch_narrow_again, for the latter, whose scores are infinite,
// the caller asks the corpus itself. Unit vectors of 768: the margin is 1.3e-3, within which
// a sixth more rows than the k best are. The scores are those of search_top_kernel.
//
// Us in a stream, k = 10, score_topk and this, 250000 rows of 768: 1 query 138, 79; 16
// 159, 83; 17 161, 100; 128 239, 102; 256 355, 126; 20000 rows of 384: 1 14, 13; 16 37,
// 14; 256 41, 24.
//
// Rows and queries lie in the order of the matrix cores' operands: blocks of 16 rows
// by 32 columns, [ceil(N / 16)][KP / 32][64 lanes][8 numbers], lane l with row l % 16
// and columns l / 16 * 8 on. A block is 1 KiB that goes to LDS, and from there to the
// lanes, as it lies. Rows past the last are the last one again.
#include "search_rows.h"

#include <algorithm>
#include <limits.h>
#include <type_traits>

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef unsigned short u16;

extern __shared__ __attribute__((aligned(16))) char smem[];

#define NS_UNSURE INT_MIN
#define NS_SPANS 1024  // spans of rows that a query may have to look into
#define NS_LIST 1024   // groups that may be near
#define NS_CAP 256     // groups that are scored
#define NS_AGAIN 32    // queries that are asked again in a launch
#define NS_LISTS 256   // lists of their best rows, a workgroup each
#define NS_PIECE 128   // groups that these score at a time

// ---- rows -------------------------------------------------------------------
// Bits of the largest magnitude of n numbers, n % 4 == 0, into *most (0 ahead):
// whole numbers of the same order, infinity and NaN the largest.
__global__ void __launch_bounds__(256)
narrow_most_kernel(const float* __restrict__ x, long n, int* __restrict__ most) {
  const long step = (long)gridDim.x * 1024;
  int m = 0;
  for (long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4; i < n; i += step) {
    const i32x4 v = *reinterpret_cast<const i32x4*>(x + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) m = max(m, v[e] & 0x7fffffff);
  }
#pragma unroll
  for (int d = 1; d < 64; d *= 2) m = max(m, __shfl_xor(m, d));
  if ((threadIdx.x & 63) == 0) atomicMax(most, m);
}

// x as f16, 0 below its normal numbers, which the matrix cores need not keep
__device__ __forceinline__ _Float16 narrow_f16(float x) {
  return fabsf(x) < 0x1p-14f ? (_Float16)0.f : (_Float16)x;
}

// A wave per 16 rows. facts (bits, 0 ahead): the largest squares of |c - c'| and |c'|,
// and the sum of all |c'| squared, of rows times 2^up.
__global__ void __launch_bounds__(256)
narrow_rows_kernel(const float* __restrict__ corpus, u16* __restrict__ out,
                   long N, int K, int KP, int up, float* __restrict__ facts) {
  const int lane = threadIdx.x & 63;
  const long step = (long)gridDim.x * 4, units = (N + 15) / 16;
  float left_most = 0.f, norm_most = 0.f, all = 0.f;
  for (long unit = (long)blockIdx.x * 4 + (threadIdx.x >> 6); unit < units;
       unit += step) {
    const long row = min(unit * 16 + (lane & 15), N - 1);
    float left = 0.f, norm = 0.f;
#pragma unroll 2
    for (int c = 0; c < KP; c += 32) {
      const int at = c + (lane >> 4) * 8;
      f16x8 o;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        f32x4 x = {0.f, 0.f, 0.f, 0.f};
        if (at + h * 4 < K)
          x = *reinterpret_cast<const f32x4*>(corpus + row * K + at + h * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = ldexpf(x[e], up);
          const _Float16 n = narrow_f16(v);
          const float f = (float)n;
          left = fmaf(v - f, v - f, left);
          norm = fmaf(f, f, norm);
          o[h * 4 + e] = n;
        }
      }
      *reinterpret_cast<f16x8*>(out + (unit * KP + c) * 16 + lane * 8) = o;
    }
    left = lanes_sum<16>(lanes_sum<32>(left));
    norm = lanes_sum<16>(lanes_sum<32>(norm));
    left_most = fmaxf(left_most, left);
    norm_most = fmaxf(norm_most, norm);
    all += norm;
  }
  left_most = wave_reduce_max(left_most);
  norm_most = wave_reduce_max(norm_most);
  all = wave_reduce_sum(all) * 0.25f;  // four lanes have a row's
  if (lane == 0) {
    atomicMax(reinterpret_cast<int*>(facts), __builtin_bit_cast(int, left_most));
    atomicMax(reinterpret_cast<int*>(facts) + 1,
              __builtin_bit_cast(int, norm_most));
    atomicAdd(facts + 2, all);
  }
}

// ---- queries ------------------------------------------------------------------
struct NarrowRows {
  const u16* rows;
  int N, K, KP, up;
  float error, norm;  // |c - c'| and |c'| at most, of rows times 2^up
};

// A query as f16, by one wave: times the power of two that brings its largest number to
// 2^13, zeros behind K, as put(column, four numbers) for KP columns; first as it is to
// `copy`, from where it is read again (q may be memory of the host). The margin (see
// above) of products of the scaled numbers, infinite where it cannot be said.
template <class F>
__device__ __forceinline__ float narrow_query(const float* q, float* copy,
                                              const NarrowRows& c, F put) {
  const int lane = threadIdx.x & 63;
  auto four = [&](int i) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(copy + min(i, c.K - 4));
    return i < c.K ? x : f32x4{0.f, 0.f, 0.f, 0.f};
  };
  int bits = 0;
#pragma unroll 3
  for (int i = lane * 4; i < c.K; i += 256) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(q + i);
    *reinterpret_cast<f32x4*>(copy + i) = x;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      bits = max(bits, __builtin_bit_cast(int, (float)x[e]) & 0x7fffffff);
  }
#pragma unroll
  for (int d = 1; d < 64; d *= 2) bits = max(bits, __shfl_xor(bits, d));
  const bool sure = bits < 0x7f800000;
  const int up = sure && bits > 0
                     ? min(13 - ilogbf(__builtin_bit_cast(float, bits)), 120)
                     : 0;
  float whole = 0.f, left = 0.f, norm = 0.f;
#pragma unroll 3
  for (int i = lane * 4; i < c.KP; i += 256) {
    const f32x4 x = four(i);
    u16 o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float v = sure ? ldexpf(x[e], up) : 0.f;
      const _Float16 h = narrow_f16(v);
      const float f = (float)h;
      whole = fmaf(v, v, whole);
      left = fmaf(v - f, v - f, left);
      norm = fmaf(f, f, norm);
      o[e] = __builtin_bit_cast(u16, h);
    }
    put(i, *reinterpret_cast<const i32x2*>(o));
  }
  whole = sqrtf(wave_reduce_sum(whole));
  left = sqrtf(wave_reduce_sum(left));
  norm = sqrtf(wave_reduce_sum(norm));
  // (products that float32 cannot hold are not for this way)
  const float size = ldexpf(whole * 0x1p-20f, -up) * ldexpf(c.norm, -c.up);
  if (!sure || !(size < 0x1p100f) || !(size > 0x1p-100f)) return INFINITY;
  // a thousandth more than what the sums of squares may be off
  return 2.002f * (whole * c.error + left * c.norm +
                   (c.K + 64) * 0x1p-23f * norm * c.norm);
}

// Queries in blocks as the rows, a wave each: of 16 FN queries lane r has query FN r + f
// in the f-th block. Zeros past Q. q may be memory of the host: one launch takes it to
// the GPU and makes what is asked of it.
__global__ void __launch_bounds__(256)
narrow_queries_kernel(const float* q, float* copy, u16* __restrict__ out,
                      float* __restrict__ margin, int* __restrict__ spent,
                      const NarrowRows c, int Q, int FN) {
  if (blockIdx.x == 0 && threadIdx.x < NS_AGAIN) spent[threadIdx.x] = 0;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int block = row / (16 * FN) * FN + row % FN, r = row / FN % 16;
  auto at = [&](int i) {
    return reinterpret_cast<i32x2*>(out + ((long)block * c.KP + (i & ~31)) * 16 +
                                    ((i >> 3 & 3) * 16 + r) * 8 + (i & 4));
  };
  if (row < Q) {
    const float m =
        narrow_query(q + (long)row * c.K, copy + (long)row * c.K, c,
                     [&](int i, i32x2 v) { *at(i) = v; });
    if ((threadIdx.x & 63) == 0) margin[row] = m;
  } else {
    for (int i = (threadIdx.x & 63) * 4; i < c.KP; i += 256) *at(i) = {0, 0};
  }
}

// ---- a few queries -------------------------------------------------------------
// Up to 16 queries: groups[(N + 3) / 4, Q], of every four rows the largest product,
// and spans[Q, waves], of a wave's rows. A wave has every W-th sixteen of rows, so
// that all read beside each other, and a ring of its own in LDS for their chunks of 64
// columns, filled R - 1 chunks ahead: no barriers, counted waits. The queries are in
// LDS as a whole. Bound by reading the rows: 250000 of 768 66 us, 5.8 TB/s.
constexpr int NF_WAVES = 8, NF_RING = 6;
static int narrow_few_lds(int KP) {
  return KP * 32 + NF_WAVES * NF_RING * 2048;
}

// 1 KiB from a pointer that all lanes share
__device__ __forceinline__ void narrow_copy(const u16* src, char* dst) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) unsigned int*)(
          src + (threadIdx.x & 63) * 8),
      (__attribute__((address_space(3))) unsigned int*)dst, 16, 0, 0);
}

__global__ void __launch_bounds__(NF_WAVES * 64)
narrow_few_kernel(const u16* __restrict__ rows, const u16* __restrict__ q16,
                  float* __restrict__ groups, float* __restrict__ spans, int Q,
                  int N, int KP) {
  constexpr int R = NF_RING;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int nch = KP / 64, W = gridDim.x * NF_WAVES;
  const int own = wid * gridDim.x + blockIdx.x;  // among all waves
  const int units = (N + 15) / 16;
  const int mine = own < units ? (units - own + W - 1) / W : 0;
  char* ring = smem + KP * 32 + wid * (R * 2048);

  // to be copied next: a chunk of a unit's
  const u16* src = rows + (long)own * KP * 16;
  const long hop = (long)(W - 1) * KP * 16;
  int chunk = 0;
  auto issue = [&](int slot) {
#pragma unroll
    for (int p = 0; p < 2; ++p)
      narrow_copy(src + p * 512, ring + slot * 2048 + p * 1024);
    src += 1024;
    if (++chunk == nch) {
      chunk = 0;
      src += hop;
    }
  };
  const int total = mine * nch;
  for (int c = 0; c < R - 1 && c < total; ++c) issue(c);
  for (int c = wid; c < nch * 2; c += NF_WAVES)
    narrow_copy(q16 + c * 512, smem + c * 1024);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  float top = -INFINITY;
  int slot = 0, left = total;
  const int G = (N + 3) / 4;
  for (int u = own; u < units; u += W) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int c = 0; c < nch; ++c, --left) {
      if (left > R - 1) {
        issue(slot == 0 ? R - 1 : slot - 1);
        asm volatile("s_waitcnt vmcnt(%0)" ::"i"((R - 1) * 2) : "memory");
      } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      const char* b = ring + slot * 2048 + lane * 16;
      const char* y = smem + c * 2048 + lane * 16;
#pragma unroll
      for (int h = 0; h < 2; ++h)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(
            *reinterpret_cast<const f16x8*>(b + h * 1024),
            *reinterpret_cast<const f16x8*>(y + h * 1024), acc, 0, 0, 0);
      // the slot is read before the wave fills it again
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      slot = slot == R - 1 ? 0 : slot + 1;
    }
    const float m = fmaxf(fmaxf(acc[0], acc[1]), fmaxf(acc[2], acc[3]));
    top = fmaxf(top, m);
    if (r < Q && u * 4 + g < G) groups[(long)(u * 4 + g) * Q + r] = m;
  }
  top = lanes_max<16>(lanes_max<32>(top));
  if (lane < Q && lane < 16) spans[(long)lane * W + own] = top;
}

// ---- batches -------------------------------------------------------------------
// groups[(N + 3) / 4, cols] and spans[cols, 2 tiles] of a half of a tile's rows, cols
// the queries in whole tiles. A workgroup stays on its CU and makes one tile of 32 FM
// rows by 32 FN queries after the other, 4 waves with 16 FM x 16 FN each: the sums are
// all 256 accumulation registers at FM = FN = 8. Steps of 32 columns go through two
// rings in LDS, over the edges of tiles; while the matrix cores work on a step the
// operands of the next are read. Queries come from the L2; rows come from memory and
// are copied more steps ahead. Copies of a wave come back in order, so two waves copy
// rows and two queries. A lane has FN neighbouring queries, so that what leaves the
// registers is whole lines; these stores drain during the next tile (vmcnt counts in
// order).
// 250000 rows of 768 and 256 queries 102 us, which is what the matrix cores and LDS do
// not overlap (without its stores 98); 128 84, of which the 32 MB of groups are 15.
// (slots of the rings; 160 KiB, and no more copies than vmcnt counts)
constexpr int nb_queries(int FM, int FN) {
  return FM == 8 ? (FN == 8 ? 3 : 4) : FN == 8 ? 6 : 8;
}
constexpr int nb_rows(int FM, int FN) {
  return FM == 8 ? (FN == 8 ? 7 : 8) : FN == 8 ? 8 : 12;
}
constexpr int nb_lds(int FM, int FN) {
  return nb_queries(FM, FN) * FN * 2048 + nb_rows(FM, FN) * FM * 2048;
}

__device__ __forceinline__ void nb_copy(const char* from, int lane_at, int to) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %2"
      :
      : "s"(to), "v"(lane_at), "s"(from)
      : "memory");
}
template <int N>
__device__ __forceinline__ void nb_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(N) : "memory");
}

// groups and spans are not __restrict__: the waits count a tile's stores among the
// copies in assembly, ahead of which they must stay.
template <int FM, int FN>
__global__ void __launch_bounds__(256, 1)
narrow_batch_kernel(const char* rows, const char* q16, float* groups,
                    float* spans, int N, int nk, int ntn) {
  constexpr int XR = nb_rows(FM, FN), XB = FM * 2048;
  constexpr int WR = nb_queries(FM, FN), WB = FN * 2048, X0 = WR * WB;
  constexpr int STORES = FM * FN / 4 + FN / 4, MOST = FM > FN ? FM : FN;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int mh = wid >> 1, nh = wid & 1;  // the wave's half of rows, queries
  const int units = (N + 15) / 16, ntm = (units + 2 * FM - 1) / (2 * FM);
  const int cols = ntn * 32 * FN;

  // every XCD has a run of tiles of its own, its workgroups take turns
  const int tiles = ntm * ntn, per = gridDim.x >> 3, xcd = blockIdx.x & 7;
  const int t0 = (int)((long)tiles * xcd / 8) + (blockIdx.x >> 3);
  const int t1 = (int)((long)tiles * (xcd + 1) / 8);
  if (t0 >= t1) return;

  // ---- copies: waves 0 and 1 of queries, FN a step, 2 and 3 of rows, FM a step
  const bool of_rows = mh != 0;
  const long block = (long)nk * 1024;  // of a 16 of rows
  const char* from[MOST];
  // the step with which every tile begins; it goes round from there
  const int turn = (int)((unsigned)(blockIdx.x >> 3) * 5 % (unsigned)nk);
  int ct = t0, ck = turn, lane_at = lane * 16 + turn * 1024;
  auto tile = [&]() {
    const int tm = ct / ntn, tn = ct - tm * ntn;
#pragma unroll
    for (int i = 0; i < MOST; ++i)
      from[i] = of_rows ? rows + min(tm * (2 * FM) + nh * FM + i, units - 1) * block
                        : q16 + (tn * 2 + nh) * FN * block + min(i, FN - 1) * block;
  };
  tile();
  const int own = of_rows ? X0 + nh * FM * 1024 : nh * FN * 1024;
  auto copy = [&](int slot, int i) {  // i-th of this wave's
    if ((i < FM && i < FN) || (of_rows ? i < FM : i < FN))
      nb_copy(from[i], lane_at, own + slot + i * 1024);
  };
  // behind the last tile it is copied again, for nobody
  auto copied = [&]() {
    lane_at += 1024;
    if (++ck == nk) {
      ck = 0;
      lane_at = lane * 16;
    }
    if (ck == turn) {
      if (ct + per < t1) ct += per;
      tile();
    }
  };
  for (int s = 0; s < (of_rows ? XR : WR); ++s) {
#pragma unroll
    for (int i = 0; i < MOST; ++i) copy(s * (of_rows ? XB : WB), i);
    copied();
  }

  // ---- products
  f16x8 xa[FM], wa[FN], xb[FM], wb[FN];
  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM * FN; ++i) acc[i / FN][i % FN] = {0.f, 0.f, 0.f, 0.f};
  const int xread = X0 + mh * FM * 1024 + lane * 16;
  const int wread = nh * FN * 1024 + lane * 16;
  auto read = [&](f16x8(&x)[FM], f16x8(&w)[FN], int xat, int wat, int i) {
    if (i < FN)
      w[i] = *reinterpret_cast<const f16x8*>(smem + wat + wread + i * 1024);
    else
      x[i - FN] = *reinterpret_cast<const f16x8*>(smem + xat + xread +
                                                  (i - FN) * 1024);
  };
  if (of_rows) nb_wait<(XR - 1) * FM>();
  else nb_wait<(WR - 1) * FN>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < FM + FN; ++i) read(xa, wa, 0, 0, i);

  int xslot = 0, wslot = 0, puts = 0;  // steps for which stores may be in flight
  auto step = [&](auto start, f16x8(&x)[FM], f16x8(&w)[FN], f16x8(&xn)[FM],
                  f16x8(&wn)[FN]) {
    constexpr bool START = decltype(start)::value;
    // the next step is there, and this one's slots are read by all
    if (of_rows) {
      if (puts > 0) nb_wait<(XR - 2) * FM + STORES>();
      else nb_wait<(XR - 2) * FM>();
    } else {
      if (puts > 0) nb_wait<(WR - 2) * FN + STORES>();
      else nb_wait<(WR - 2) * FN>();
    }
    --puts;
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const int xnext = xslot == (XR - 1) * XB ? 0 : xslot + XB;
    const int wnext = wslot == (WR - 1) * WB ? 0 : wslot + WB;
    const int slot = of_rows ? xslot : wslot;
    constexpr int READS = FM + FN, EVERY = (FM * FN - 4) / READS;
    constexpr int GAP = FM * FN / MOST;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < FM * FN; ++s) {
      f32x4& c = acc[s / FN][s % FN];
      // the sums begin here, in assembly because the compiler would keep them
      // elsewhere and move them
      if constexpr (START)
        asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0"
                     : "+a"(c)
                     : "v"(x[s / FN]), "v"(w[s % FN]));
      else
        c = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[s / FN], w[s % FN], c, 0,
                                                   0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (s % EVERY == EVERY / 2 && s / EVERY < READS)
        read(xn, wn, xnext, wnext, s / EVERY);
      if (s % GAP == 1) copy(slot, s / GAP);
      __builtin_amdgcn_sched_barrier(0);
    }
    copied();
    xslot = xnext;
    wslot = wnext;
  };
  using Yes = std::true_type;
  using No = std::false_type;
  for (int t = t0; t < t1; t += per) {
    // (where a workgroup has a tile or two, code that is run once takes as long to
    // arrive as it saves)
    constexpr int FIRST = FM == 8 ? 2 : 0;
    if constexpr (FIRST) {
      step(Yes{}, xa, wa, xb, wb);
      step(No{}, xb, wb, xa, wa);
    } else {
#pragma unroll
      for (int i = 0; i < FM * FN; ++i)
        acc[i / FN][i % FN] = {0.f, 0.f, 0.f, 0.f};
    }
    for (int k = FIRST; k < nk; k += 2) {
      step(No{}, xa, wa, xb, wb);
      step(No{}, xb, wb, xa, wa);
    }

    const int tm = t / ntn;
    const int n = ((t - tm * ntn) * 2 + nh) * (16 * FN) + r * FN;
    int wide = cols;
    asm volatile("" : "+s"(wide));  // offsets are not kept over the loop
    const int here = min(FM * 32, N - tm * (FM * 32));
    const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(
        groups + (long)tm * (FM * 8) * wide, 0, (here + 3) / 4 * wide * 4,
        0x00020000);
    const int at = ((mh * (FM * 4) + g) * wide + n) * 4;
    float all[FN];
#pragma unroll
    for (int f = 0; f < FN; ++f) all[f] = -INFINITY;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      __builtin_amdgcn_sched_barrier(0);
      // the sums leave the accumulation registers here and not before
#pragma unroll
      for (int f = 0; f < FN; ++f) asm volatile("" : "+a"(acc[i][f]));
      f32x4 o[FN / 4];
#pragma unroll
      for (int f = 0; f < FN; ++f) {
        const f32x4 v = acc[i][f];
        const float m = fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3]));
        o[f >> 2][f & 3] = m;
        all[f] = fmaxf(all[f], m);
      }
#pragma unroll
      for (int h = 0; h < FN / 4; ++h)
        __builtin_amdgcn_raw_buffer_store_b128(
            __builtin_bit_cast(i32x4, o[h]), out, at + i * 16 * wide + h * 16,
            0, 0);
    }
    // of the four lanes that have these queries each keeps a quarter of them
    auto most = [](float a, float b, auto swap) {
      const i32x2 v =
          swap(__builtin_bit_cast(int, a), __builtin_bit_cast(int, b));
      const int x = v[0], y = v[1];
      return fmaxf(__builtin_bit_cast(float, x), __builtin_bit_cast(float, y));
    };
    auto halves = [](int a, int b) -> i32x2 {
      return __builtin_amdgcn_permlane32_swap(a, b, false, false);
    };
    auto quarters = [](int a, int b) -> i32x2 {
      return __builtin_amdgcn_permlane16_swap(a, b, false, false);
    };
    float two[FN / 2], one[FN / 4];
#pragma unroll
    for (int f = 0; f < FN / 2; ++f)
      two[f] = most(all[f], all[FN / 2 + f], halves);
#pragma unroll
    for (int f = 0; f < FN / 4; ++f) {
      one[f] = most(two[f], two[FN / 4 + f], quarters);
      if (mh * (FM * 16) >= here) one[f] = -INFINITY;  // it has no rows
    }
#pragma unroll
    for (int f = 0; f < FN / 4; ++f)
      spans[(long)(n + g * (FN / 4) + f) * (ntm * 2) + tm * 2 + mh] = one[f];
    puts = (of_rows ? XR : WR) - 1;
  }
  // nothing is in flight to LDS that the next workgroup may have
  nb_wait<0>();
}

// ---- choice -------------------------------------------------------------------
// Where the products are: groups[G, ld], of query q in column q, and spans[., S]; span
// s has the groups s A + j / A B + j % A for j < each.
struct NarrowMost {
  const float *groups, *spans, *margin;
  float* limit;  // of a query that is not answered: its best rows' groups are above
  long ld;
  int S, A, B, each, G;
  __device__ int group(int s, int j) const { return s * A + j / A * B + j % A; }
};

// Score and place as one number: the larger score, then the smaller row, is the larger.
__device__ __forceinline__ unsigned long long narrow_key(float v, int row) {
  return ((unsigned long long)f32_to_ord(v) << 32) | (unsigned int)~row;
}

// Keys of the rows r0 to r0 + 3, by one wave; 0 past the last.
__device__ __forceinline__ void narrow_score(const float* query,
                                             const float* corpus, int r0, int N,
                                             int K, unsigned long long* keys) {
  const int lane = threadIdx.x & 63;
  float s[4];
  search_dot(query, corpus, r0, N, K, s);
  if (lane < 4) {
    const float v = lane == 0 ? s[0] : lane == 1 ? s[1] : lane == 2 ? s[2] : s[3];
    keys[lane] = r0 + lane < N ? narrow_key(v, r0 + lane) : 0ull;
  }
}

// A workgroup per query. The k-th largest of 64 shares of the spans bounds the k-th
// largest group from below; the spans within the margin of it are looked into, where
// the same is found of their groups, then the k-th largest itself. Rows of groups
// within the margin of that are scored in plain float32; equals go by place. k <= 60.
// A chain of loads and barriers, and of 256 queries 44 MB of rows: under the profiler, of
// 250000 rows of 768, 1 query 7.1 us, 256 16.1 (9.3 and 18.0 with the 64 shares' ranks
// found by one wave, and the spans read again once there is a bound).
__global__ void __launch_bounds__(1024)
narrow_top_kernel(const NarrowMost o, const float* __restrict__ q,
                  const float* __restrict__ corpus,
                  float* __restrict__ out_v, int* __restrict__ out_i, int N,
                  int K, int k) {
  __shared__ float top[16][64], thresh;
  __shared__ int nspan, nlist, ncand, ranks[64];
  __shared__ int span[NS_SPANS], list[NS_LIST], cand[NS_CAP];
  __shared__ float near[NS_LIST];
  __shared__ unsigned long long rows[NS_CAP * 4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int me = blockIdx.x;
  const float margin = o.margin[me];
  float* ov = out_v + (long)me * k;
  int* oi = out_i + (long)me * k;
  auto unsure = [&](float limit) {
    if (tid < k) {
      ov[tid] = limit;
      oi[tid] = NS_UNSURE;
    }
    if (tid == 0) o.limit[me] = limit;
  };
  if (!(margin < INFINITY)) return unsure(INFINITY);
  if (tid == 0) nspan = nlist = ncand = 0;
  if (tid < 64) ranks[tid] = 0;
  // the k-th largest of 64 shares' largest, of all threads' m
  auto bound = [&](float m) {
    top[wid][lane] = m;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 16; ++w) m = fmaxf(m, top[w][lane]);
    // a wave compares with four of the shares
    int rank = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int j = wid * 4 + i;
      const float v = __builtin_bit_cast(
          float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, m), j));
      rank += v > m || (v == m && j < lane);
    }
    if (rank > 0) atomicAdd(&ranks[lane], rank);
    __syncthreads();
    if (tid < 64) {
      if (ranks[lane] == k - 1) thresh = m;
      ranks[lane] = 0;
    }
    __syncthreads();
    return thresh;
  };

  float m = -INFINITY, first[2];
  const float* spans = o.spans + (long)me * o.S;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int s = tid + i * 1024;
    first[i] = s < o.S ? spans[s] : -INFINITY;
    m = fmaxf(m, first[i]);
  }
#pragma unroll 2
  for (int s = tid + 2048; s < o.S; s += 1024) m = fmaxf(m, spans[s]);
  float least = bound(m);
  if (m >= least - margin)
    for (int s = tid, i = 0; s < o.S; s += 1024, ++i) {
      const float v = i == 0 ? first[0] : i == 1 ? first[1] : spans[s];
      if (v >= least - margin) {
        const int to = atomicAdd(&nspan, 1);
        if (to < NS_SPANS) span[to] = s;
      }
    }
  __syncthreads();
  if (nspan > NS_SPANS) return unsure(least - margin);

  const int items = nspan * o.each;
  // those within the margin, and the largest number of this thread's
  auto gather = [&]() {
    float m = -INFINITY;
    for (int i = tid; i < items; i += 1024) {
      const int at = o.group(span[i / o.each], i % o.each);
      if (at >= o.G) continue;
      const float v = o.groups[at * o.ld + me];
      m = fmaxf(m, v);
      if (v >= least - margin) {
        const int to = atomicAdd(&nlist, 1);
        if (to < NS_LIST) {
          list[to] = at;
          near[to] = v;
        }
      }
    }
    __syncthreads();
    return m;
  };
  m = gather();
  // spans with many of them: a better bound is found among their groups
  if (nlist > NS_LIST) {
    __syncthreads();
    if (tid == 0) nlist = 0;
    least = fmaxf(least, bound(m));
    gather();
  }
  const int n = nlist;
  if (n > NS_LIST) return unsure(least - margin);
  const float own = tid < n ? near[tid] : -INFINITY;
  if (n > 2 * NS_CAP) {  // (ranks of 750 take 20 us, a bound of them 1)
    least = fmaxf(least, bound(own));
    if (own >= least - margin) atomicAdd(&ncand, 1);
    __syncthreads();
    if (ncand > 2 * NS_CAP) return unsure(least - margin);
    __syncthreads();
    if (tid == 0) ncand = 0;
  }
  // (fewer groups than k are all that there are)
  if (tid == 0) thresh = -INFINITY;
  __syncthreads();
  if (tid < n) {
    int rank = 0;
    for (int j = 0; j < n; ++j)
      rank += near[j] > own || (near[j] == own && j < tid);
    if (rank == k - 1) thresh = own;
  }
  __syncthreads();
  if (tid < n && own >= thresh - margin) {
    const int to = atomicAdd(&ncand, 1);
    if (to < NS_CAP) cand[to] = list[tid];
  }
  __syncthreads();
  const int take = ncand;
  if (take > NS_CAP) return unsure(thresh - margin);

  const float* query = q + (long)me * K;
  for (int c = wid; c < take; c += 16)
    narrow_score(query, corpus, cand[c] * 4, N, K, rows + c * 4);
  __syncthreads();
  if (tid >= take * 4) return;
  const unsigned long long key = rows[tid];
  int r = 0;
#pragma unroll 8
  for (int j = 0; j < take * 4; ++j) r += rows[j] > key;
  if (key != 0 && r < k) {
    ov[r] = ord_to_f32((unsigned int)(key >> 32));
    oi[r] = (int)~(unsigned int)key;
  }
}

// ---- queries beside many rows that are nearly as good ---------------------------
// A query that narrow_top_kernel left for them, by NS_LISTS workgroups: each looks
// into every NS_LISTS-th span, scores the groups above the limit and keeps the k best
// rows, largest first, as keys, 0 behind them. spent counts the groups of a query;
// above `most` (the corpus itself is read in less) it is left unanswered.
// Bound by reading these rows, and by the launches where they are few thousands: a search
// of 250000 rows of 768 with a question beside 3000 equal ones, us, all questions asked
// of the corpus and this: one 173 and 136 (101 without such rows), 256 450 and 257 (218);
// 20 of 256 292.
struct NarrowAgain {
  int who[NS_AGAIN];
};

__global__ void __launch_bounds__(1024)
narrow_again_kernel(const NarrowMost o, const NarrowAgain a,
                    const float* __restrict__ q,
                    const float* __restrict__ corpus,
                    unsigned long long* __restrict__ lists, int* spent, int most,
                    int N, int K, int k) {
  __shared__ unsigned long long keys[64 + NS_PIECE * 4];  // the best, new ones
  __shared__ int list[1024], near, before;
  const int tid = threadIdx.x;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int me = a.who[blockIdx.y], first = blockIdx.x;
  const float limit = o.limit[me];
  const float* query = q + (long)me * K;
  const float* spans = o.spans + (long)me * o.S;
  if (tid < 64) keys[tid] = 0;
  const int items =
      limit < INFINITY && first < o.S
          ? ((o.S - 1 - first) / NS_LISTS + 1) * o.each
          : 0;
  for (int i0 = 0; i0 < items; i0 += 1024) {
    if (tid == 0) near = 0;
    __syncthreads();
    const int i = i0 + tid, s = first + i / o.each * NS_LISTS;
    if (i < items && spans[s] >= limit) {
      const int at = o.group(s, i % o.each);
      if (at < o.G && o.groups[at * o.ld + me] >= limit)
        list[atomicAdd(&near, 1)] = at;
    }
    __syncthreads();
    const int take = near;
    if (tid == 0) before = take > 0 ? atomicAdd(spent + blockIdx.y, take) : 0;
    __syncthreads();
    if (before + take > most) break;
    for (int c0 = 0; c0 < take; c0 += NS_PIECE) {
      const int piece = min(take - c0, NS_PIECE), all = 64 + piece * 4;
      for (int c = wid; c < piece; c += 16)
        narrow_score(query, corpus, list[c0 + c] * 4, N, K, keys + 64 + c * 4);
      __syncthreads();
      const unsigned long long key = tid < all ? keys[tid] : 0;
      int r = 0;
#pragma unroll 8
      for (int j = 0; j < all; ++j) r += keys[j] > key;
      __syncthreads();
      if (key != 0 && r < k) keys[r] = key;
      __syncthreads();
    }
  }
  __syncthreads();
  if (tid < k)
    lists[((long)blockIdx.y * NS_LISTS + first) * k + tid] = keys[tid];
}

// The k best of a query's lists, a thread each.
__global__ void __launch_bounds__(NS_LISTS)
narrow_pick_kernel(const NarrowAgain a,
                   const unsigned long long* __restrict__ lists,
                   const int* __restrict__ spent, int most,
                   float* __restrict__ out_v, int* __restrict__ out_i, int k) {
  __shared__ unsigned long long top[2][NS_LISTS / 64];
  if (spent[blockIdx.x] > most) return;
  const long me = a.who[blockIdx.x];
  const unsigned long long* mine =
      lists + ((long)blockIdx.x * NS_LISTS + threadIdx.x) * k;
  unsigned long long key = mine[0];
  for (int r = 0, at = 0; r < k; ++r) {
    unsigned long long m = key;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
      const unsigned long long other = __shfl_xor(m, d);
      m = other > m ? other : m;
    }
    if ((threadIdx.x & 63) == 0) top[r & 1][threadIdx.x >> 6] = m;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NS_LISTS / 64; ++w)
      m = top[r & 1][w] > m ? top[r & 1][w] : m;
    if (m == 0) return;  // there are none
    if (key == m) {
      out_v[me * k + r] = ord_to_f32((unsigned int)(m >> 32));
      out_i[me * k + r] = (int)~(unsigned int)m;
      key = ++at < k ? mine[at] : 0;
    }
  }
}

// ---- launches -----------------------------------------------------------------
extern "C" void launch_narrow_most(const float* x, long n, int* most,
                                   hipStream_t stream) {
  hipLaunchKernelGGL(narrow_most_kernel, dim3(std::min(n / 4096 + 1, 2048L)),
                     dim3(256), 0, stream, x, n, most);
}

extern "C" void launch_narrow_rows(const float* corpus, void* out, long N,
                                   int K, int KP, int up, float* facts,
                                   hipStream_t stream) {
  hipLaunchKernelGGL(narrow_rows_kernel, dim3(std::min(N / 64 + 1, 4096L)),
                     dim3(256), 0, stream, corpus, (u16*)out, N, K, KP, up,
                     facts);
}

namespace {

// Where things lie beside the operands.
struct NarrowPlan {
  int QP, fm, fn, grid;  // fn 1: a few queries
  long copy, q16, margin, limit, spent, groups, spans, bytes;
  NarrowMost most;
};

NarrowPlan narrow_plan(int Q, int N, int K, int KP) {
  NarrowPlan p = {};
  p.fn = Q <= 16 && KP <= 1536 ? 1 : Q <= 128 ? 4 : 8;
  const int tile = p.fn == 1 ? 16 : 32 * p.fn;
  p.QP = (Q + tile - 1) / tile * tile;
  NarrowMost& o = p.most;
  o.G = (N + 3) / 4;
  if (p.fn == 1) {
    const int units = (N + 15) / 16;
    p.grid = std::min(units, 256);
    o.S = p.grid * NF_WAVES;
    o.A = 4;
    o.B = 4 * o.S;
    o.each = (units + o.S - 1) / o.S * 4;
    o.ld = Q;
  } else {
    // Tiles of 256 rows that leave half of the CUs without one are halved: 200 sizes
    // of 128 to 4096 columns, time by 128 rows over that by 256, up to 128 tiles 0.57
    // to 0.95 (1000 x 4096 1.01), 129 to 256, where the halves are a second round,
    // 0.88 to 1.02 of 128 columns and 0.95 to 1.23 beyond, above 0.95 to 1.21.
    const long tiles = (N + 255L) / 256 * (p.QP / tile);
    p.fm = tiles <= 128 ? 4 : 8;
    o.S = (N + 32 * p.fm - 1) / (32 * p.fm) * 2;
    o.A = o.each = p.fm * 4;
    o.ld = p.QP;
  }
  auto place = [&](long bytes) {
    const long at = p.bytes;
    p.bytes += (bytes + 255) / 256 * 256;
    return at;
  };
  p.copy = place((long)Q * K * 4);
  p.q16 = place((long)p.QP * KP * 2);
  p.margin = place((long)Q * 4);
  p.limit = place((long)Q * 4);
  p.spent = place(NS_AGAIN * 4);
  p.spans = place(o.S * o.ld * 4);
  p.groups = place(o.G * o.ld * 4);
  return p;
}

NarrowMost narrow_most(const NarrowPlan& p, char* space) {
  NarrowMost o = p.most;
  o.groups = (const float*)(space + p.groups);
  o.spans = (const float*)(space + p.spans);
  o.margin = (const float*)(space + p.margin);
  o.limit = (float*)(space + p.limit);
  return o;
}

}  // namespace

// Bytes that launch_narrow_topk needs beside its operands, 0 where it does not take
// these sizes (tiles are counted, and groups of a tile addressed, in 32 bits).
extern "C" long narrow_bytes(long Q, long N, long K, long KP) {
  if (Q < 1 || Q >= 1L << 20 || N < 1 || N > (1L << 31) - 1024 || K < 4 ||
      K % 4 || KP % 64 || KP < 128 || KP < K || KP > 1L << 16 ||
      (N + 127) / 128 * ((Q + 127) / 128) >= 1L << 30)
    return 0;
  return narrow_plan((int)Q, (int)N, (int)K, (int)KP).bytes;
}

// rows: of narrow_rows_kernel, with its up and (roots of its) facts; space:
// narrow_bytes. out_v, out_i [Q, k], k <= 60 and <= N. q, out_v and out_i may be memory
// of the host that the GPU sees.
extern "C" void launch_narrow_topk(const float* q, const float* corpus,
                                   const void* rows, void* space, float* out_v,
                                   int* out_i, int Q, int N, int K, int KP,
                                   int up, float error, float norm, int k,
                                   hipStream_t stream) {
  NarrowPlan p = narrow_plan(Q, N, K, KP);
  char* at = (char*)space;
  u16* q16 = (u16*)(at + p.q16);
  float* copy = (float*)(at + p.copy);
  float *margin = (float*)(at + p.margin), *groups = (float*)(at + p.groups),
        *spans = (float*)(at + p.spans);
  const NarrowRows c = {(const u16*)rows, N, K, KP, up, error, norm};
  hipLaunchKernelGGL(narrow_queries_kernel, dim3(p.QP / 4), dim3(256), 0,
                     stream, q, copy, q16, margin, (int*)(at + p.spent), c, Q,
                     p.fn);
  if (p.fn == 1)
    hipLaunchKernelGGL(narrow_few_kernel, dim3(p.grid), dim3(NF_WAVES * 64),
                       narrow_few_lds(KP), stream, c.rows, q16, groups, spans,
                       Q, N, KP);
#define NS(M, F)                                                             \
  hipLaunchKernelGGL((narrow_batch_kernel<M, F>), dim3(256), dim3(256),      \
                     nb_lds(M, F), stream, (const char*)c.rows,              \
                     (const char*)q16, groups, spans, N, KP / 32,            \
                     p.QP / (32 * F))
  else if (p.fm == 4 && p.fn == 4)
    NS(4, 4);
  else if (p.fm == 4)
    NS(4, 8);
  else if (p.fn == 4)
    NS(8, 4);
  else
    NS(8, 8);
#undef NS
  hipLaunchKernelGGL(narrow_top_kernel, dim3(Q), dim3(1024), 0, stream,
                     narrow_most(p, at), copy, corpus, out_v, out_i, N, K, k);
}

// How many queries launch_narrow_again takes, and the bytes of `lists` for each.
extern "C" int narrow_again_most() { return NS_AGAIN; }
extern "C" long narrow_again_bytes(int k) { return (long)NS_LISTS * k * 8; }

// The queries who[0] to who[n - 1] of launch_narrow_topk once more, by the same space
// and into the same out_v and out_i, if it was for near rows that they were left
// unanswered, up to a share of the corpus (half of it over all of them, beyond which
// the corpus itself is read in less). Once for a launch_narrow_topk.
extern "C" void launch_narrow_again(const float* corpus, void* space,
                                    const int* who, int n,
                                    unsigned long long* lists, float* out_v,
                                    int* out_i, int Q, int N, int K, int KP,
                                    int k, hipStream_t stream) {
  const NarrowPlan p = narrow_plan(Q, N, K, KP);
  char* at = (char*)space;
  int* spent = (int*)(at + p.spent);
  NarrowAgain a = {};
  for (int i = 0; i < n; ++i) a.who[i] = who[i];
  const int most = N / 8 / n;
  hipLaunchKernelGGL(narrow_again_kernel, dim3(NS_LISTS, n), dim3(1024), 0,
                     stream, narrow_most(p, at), a, (const float*)(at + p.copy),
                     corpus, lists, spent, most, N, K, k);
  hipLaunchKernelGGL(narrow_pick_kernel, dim3(n), dim3(NS_LISTS), 0, stream, a,
                     lists, spent, most, out_v, out_i, k);
}
