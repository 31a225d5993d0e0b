// kNN search kernels replacing faiss-gpu (reference rag/search.py:231-399):
// chunked radix-select top-k over a score matrix,
// and packed-binary Hamming scoring for the ubinary precision path.
//
// Pipeline (python side, rag/search.py here):
//   a few queries: search_few_kernel multiplies and leaves its runs' best rows,
//   topk_regs_kernel joins them
//   batches: score.hip leaves the best of every four rows, search_top_kernel
//   scores the best fours again
//   else: scores_chunk = Q @ C_chunk^T by the library, topk_chunk_kernel ->
//   per-chunk candidates, and again over these (with idx indirection)
//
// topk_regs_kernel takes small k (the caller's choice); beyond,
// topk_chunk_kernel: one 256-thread block per (query, chunk). Two-round
// 8-bit radix select over monotonic uint32 keys finds a threshold, a
// compact pass gathers candidates (cap 2048) into LDS, a bitonic sort
// orders them, and the top k (vals + indices) are written out.
#include "search_rows.h"

#define TK_CAP 2048  // candidate buffer (vals+idx) in LDS

// scores: [Q, N] f32. in_idx: optional [Q, N] int32 (indirection from a
// previous candidate round); out: [Q, nchunks, k] vals f32 + idx int32.
__global__ void __launch_bounds__(256)
topk_chunk_kernel(const float* __restrict__ scores,
                  const int* __restrict__ in_idx,
                  float* __restrict__ out_v, int* __restrict__ out_i,
                  long N, int chunk, int k, int nchunks) {
  __shared__ unsigned int hist[256];
  __shared__ unsigned int cnt_hi, thresh, ncand;
  __shared__ unsigned int cand_u[TK_CAP];
  __shared__ int cand_i[TK_CAP];

  const int q = blockIdx.y;
  const int c = blockIdx.x;
  const long c0 = (long)c * chunk;
  const long c1 = min(c0 + chunk, N);
  const float* row = scores + (long)q * N;

  // ---- round 1: top-8-bit histogram ----------------------------------
  if (threadIdx.x < 256) hist[threadIdx.x] = 0;
  __syncthreads();
  for (long i = c0 + threadIdx.x; i < c1; i += 256)
    atomicAdd(&hist[f32_to_ord(row[i]) >> 24], 1u);
  __syncthreads();
  // scan bins from high to low on thread 0 (256 steps, trivial)
  if (threadIdx.x == 0) {
    unsigned int acc = 0;
    int b1 = 0;
    for (int b = 255; b >= 0; --b) {
      if (acc + hist[b] >= (unsigned int)k || b == 0) { b1 = b; break; }
      acc += hist[b];
    }
    cnt_hi = acc;
    thresh = (unsigned int)b1 << 24;
  }
  __syncthreads();
  const unsigned int b1 = thresh >> 24;
  const unsigned int need2 = (unsigned int)k - cnt_hi;

  // ---- round 2: next-8-bit histogram within bin b1 --------------------
  if (threadIdx.x < 256) hist[threadIdx.x] = 0;
  __syncthreads();
  for (long i = c0 + threadIdx.x; i < c1; i += 256) {
    unsigned int u = f32_to_ord(row[i]);
    if ((u >> 24) == b1) atomicAdd(&hist[(u >> 16) & 0xffu], 1u);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned int acc = 0;
    int b2 = 0;
    for (int b = 255; b >= 0; --b) {
      if (acc + hist[b] >= need2 || b == 0) { b2 = b; break; }
      acc += hist[b];
    }
    thresh = (b1 << 24) | ((unsigned int)b2 << 16);
    ncand = 0;
  }
  __syncthreads();
  const unsigned int T = thresh;

  // ---- compact pass: gather everything with u >= T --------------------
  for (long i = c0 + threadIdx.x; i < c1; i += 256) {
    unsigned int u = f32_to_ord(row[i]);
    if (u >= T) {
      unsigned int slot = atomicAdd(&ncand, 1u);
      if (slot < TK_CAP) {
        cand_u[slot] = u;
        cand_i[slot] = in_idx ? in_idx[(long)q * N + i] : (int)i;
      }
    }
  }
  __syncthreads();
  int n = (int)min(ncand, (unsigned int)TK_CAP);
  // pad to power of two (covering k) for bitonic
  const int target = max(n, k);
  int n2 = 1;
  while (n2 < target) n2 <<= 1;
  for (int i = n + threadIdx.x; i < n2; i += 256) {
    cand_u[i] = 0;       // smallest ordinal
    cand_i[i] = -1;
  }
  __syncthreads();

  // ---- bitonic sort descending over n2 elements -----------------------
  for (int size = 2; size <= n2; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = threadIdx.x; i < n2 / 2; i += 256) {
        const int lo = 2 * i - (i & (stride - 1));
        const int hi = lo + stride;
        const bool desc = ((lo & size) == 0);
        unsigned int a = cand_u[lo], b = cand_u[hi];
        if ((a < b) == desc) {
          int ai = cand_i[lo], bi = cand_i[hi];
          cand_u[lo] = b; cand_u[hi] = a;
          cand_i[lo] = bi; cand_i[hi] = ai;
        }
      }
      __syncthreads();
    }
  }

  // ---- write top-k ----------------------------------------------------
  float* ov = out_v + ((long)q * nchunks + c) * k;
  int* oi = out_i + ((long)q * nchunks + c) * k;
  for (int i = threadIdx.x; i < k; i += 256) {
    if (i < n) {
      ov[i] = ord_to_f32(cand_u[i]);
      oi[i] = cand_i[i];
    } else {
      ov[i] = -INFINITY;
      oi[i] = -1;
    }
  }
}

// The same for chunks of up to 8192 scores and k <= 256, which a workgroup
// holds in registers: the scores are read once, and no histogram is needed as
// long as scores are not piled up (a histogram of scores of one magnitude is a
// chain of conflicting atomics). The k-th largest of the 256 threads' largest
// scores (k <= 60: of those of 64 fours of threads) bounds the k-th largest of
// the chunk from below; what reaches it is gathered and ranked, by score and,
// among equals, by place. If more than the candidate buffer holds reach it (few
// threads have all the large scores, or many scores are equal), the k-th
// largest itself is found byte by byte, and its equals are counted in the order
// of their places. (topk_chunk_kernel leaves the order of equals open.)
// Bound by reading the scores: 256 x 250000, k = 10, both rounds, 210 -> 61 us
// (4.2 TB/s); 1 x 250000, k = 5, which had 8 workgroups and now has 31, 110 ->
// 14 us. (Ranking all 256 threads' largest for any k: 167 and 35 us.) The bound
// is a poor one when k comes near the number that it is taken of: hundreds of
// scores reach it, and each is compared with all of them.
#define TR_CHUNK 8192
#define TR_CAP 1024

__global__ void __launch_bounds__(256)
topk_regs_kernel(const float* __restrict__ scores,
                 const int* __restrict__ in_idx, float* __restrict__ out_v,
                 int* __restrict__ out_i, long N, int chunk, int k,
                 int nchunks) {
  constexpr int PER = TR_CHUNK / 256;
  __shared__ __attribute__((aligned(16))) unsigned int top[256];
  __shared__ unsigned int thresh, ncand, hist[256], found, above;
  __shared__ unsigned long long key[TR_CAP];  // score, then place from the end

  const int tid = threadIdx.x;
  const int q = blockIdx.y, c = blockIdx.x;
  const long c0 = (long)c * chunk;
  const int len = (int)(min(c0 + chunk, N) - c0);
  const float* row = scores + (long)q * N + c0;

  unsigned int u[PER];
  unsigned int mine = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = tid + j * 256;
    const unsigned int v = f32_to_ord(row[min(i, len - 1)]);
    u[j] = i < len ? v : 0u;
    mine = max(mine, u[j]);
  }
  top[tid] = mine;
  if (tid == 0) ncand = 0;
  __syncthreads();
  // every rank is taken once
  if (k <= 60) {  // of 64 fours of threads, on the lanes of one wave
    if (tid < 64) {
      const unsigned int four = max(max(top[tid], top[tid + 64]),
                                    max(top[tid + 128], top[tid + 192]));
      int rank = 0;
#pragma unroll
      for (int j = 0; j < 64; ++j) {
        const unsigned int o = __builtin_amdgcn_readlane(four, j);
        rank += o > four || (o == four && j < tid);
      }
      if (rank == k - 1) thresh = four;
    }
  } else {
    int rank = 0;
#pragma unroll 8
    for (int j = 0; j < 256; ++j) {
      const unsigned int o = top[j];
      rank += o > mine || (o == mine && j < tid);
    }
    if (rank == k - 1) thresh = mine;
  }
  __syncthreads();
  unsigned int T = thresh;
  auto gather = [&](unsigned int from) {
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int i = tid + j * 256;
      if (i < len && u[j] >= from) {
        const unsigned int slot = atomicAdd(&ncand, 1u);
        if (slot < TR_CAP)
          key[slot] = ((unsigned long long)u[j] << 32) | (unsigned int)~i;
      }
    }
    __syncthreads();
  };
  gather(T);
  if (ncand > TR_CAP) {
    // the k-th largest, a byte a round: `T` its leading bytes, `want` its
    // rank among the scores that share them
    unsigned int want = k;
    T = 0;
    for (int shift = 24; shift >= 0; shift -= 8) {
      hist[tid] = 0;
      __syncthreads();
#pragma unroll
      for (int j = 0; j < PER; ++j)
        if (tid + j * 256 < len &&
            (shift == 24 || (u[j] >> (shift + 8)) == (T >> (shift + 8))))
          atomicAdd(&hist[(u[j] >> shift) & 255u], 1u);
      __syncthreads();
      if (tid == 0) {
        unsigned int sum = 0;
        int b = 255;
        for (; b > 0 && sum + hist[b] < want; --b) sum += hist[b];
        found = b;
        above = sum;
      }
      __syncthreads();
      T |= found << shift;
      want -= above;
    }
    if (tid == 0) ncand = 0;
    __syncthreads();
    // those above it (fewer than k) first, then the first `want` of its equals:
    // how many of them lie ahead of each 64 scores of a wave
    if (T != 0xffffffffu) gather(T + 1);
    const int lane = tid & 63, wid = tid >> 6;
    auto equals = [&](int j) {
      return __ballot(tid + j * 256 < len && u[j] == T);
    };
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const unsigned long long m = equals(j);
      if (lane == 0) hist[j * 4 + wid] = __popcll(m);
    }
    __syncthreads();
    if (tid < 64) {
      const unsigned int a = hist[2 * tid], b = hist[2 * tid + 1];
      unsigned int sum = a + b;
      for (int d = 1; d < 64; d *= 2) {
        const unsigned int o = __shfl_up(sum, d, 64);
        if (tid >= d) sum += o;
      }
      hist[2 * tid] = sum - a - b;
      hist[2 * tid + 1] = sum - b;
    }
    __syncthreads();
    const unsigned int first = ncand;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const unsigned long long m = equals(j);
      const unsigned int at =
          hist[j * 4 + wid] + __popcll(m & ((1ull << lane) - 1));
      if ((m >> lane & 1) && at < want)
        key[first + at] =
            ((unsigned long long)T << 32) | (unsigned int)~(tid + j * 256);
    }
    __syncthreads();
    if (tid == 0) ncand = first + want;
    __syncthreads();
  }
  const int n = (int)min(ncand, (unsigned int)TR_CAP);
  float* ov = out_v + ((long)q * nchunks + c) * k;
  int* oi = out_i + ((long)q * nchunks + c) * k;
  for (int i = tid; i < n; i += 256) {
    const unsigned long long own = key[i];
    int r = 0;
    for (int j = 0; j < n; ++j) r += key[j] > own;
    if (r < k) {
      const int at = (int)~(unsigned int)own;
      ov[r] = ord_to_f32((unsigned int)(own >> 32));
      oi[r] = in_idx ? in_idx[(long)q * N + c0 + at] : (int)(c0 + at);
    }
  }
  for (int i = n + tid; i < k; i += 256) {
    ov[i] = -INFINITY;
    oi[i] = -1;
  }
}

// Sums over the lanes of four values each; lanes 0 to 15 have the first's, then
// 16 each the third's, the second's, the fourth's.
__device__ __forceinline__ float sf_sums(const float (&s)[4]) {
  auto two = [](float a, float b, auto swap) {
    const i32x2 v = swap(__builtin_bit_cast(int, a), __builtin_bit_cast(int, b));
    const int x = v[0], y = v[1];
    return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
  };
  auto halves = [](int a, int b) -> i32x2 {
    return __builtin_amdgcn_permlane32_swap(a, b, false, false);
  };
  auto quarters = [](int a, int b) -> i32x2 {
    return __builtin_amdgcn_permlane16_swap(a, b, false, false);
  };
  float v = two(two(s[0], s[1], halves), two(s[2], s[3], halves), quarters);
  v += lane_turned<8>(v);
  v += lane_turned<4>(v);
  v += lane_turned<2>(v);
  v += lane_turned<1>(v);
  return v;
}

// Up to four queries against a corpus, in float32, and the k best rows of every
// workgroup's run for each: [Q, groups, k | 1] scores and rows, descending, equals
// by place, for topk_regs_kernel. (Of an even k the last is none, the least of
// numbers: with an even distance a few of that kernel's threads have all the lists'
// first, and k = 16 takes it 8 us longer.) A workgroup per CU; its 16 waves have a
// part of the run each and take four rows at a time, 12 KiB of 768 columns, the
// queries in LDS. A wave has the scores of 64 rows on its lanes when it looks at
// them: it ranks the first 64, and of later ones only those that are better than
// its k-th best.
// Bound by reading the corpus. us with the second launch, against the library's
// product and topk's two, one query of 768, k = 5: 250000 rows 152, 140 (5.7 TB/s
// of the product); 100000 124, 54; 30000 30, 24; 10000 19, 14; 4000 11, 12. Largest
// errors against 64 bits 2 to 10 times smaller.
#define SF_WAVES 16
template <int NC, int QN>
__global__ void __launch_bounds__(SF_WAVES * 64)
search_few_kernel(const float* __restrict__ q,
                  const float* __restrict__ corpus, float* __restrict__ out_v,
                  int* __restrict__ out_i, int Q, int N, int K, int k) {
  __shared__ f32x4 qs[QN][NC * 64];  // zeros behind K
  __shared__ unsigned long long key[QN][SF_WAVES][33], some[QN][SF_WAVES * 32];
  __shared__ unsigned int bound[QN];
  __shared__ int count[QN];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int i = tid; i < QN * NC * 64; i += SF_WAVES * 64) {
    const int at = i % (NC * 64) * 4;
    const float* from = q + (long)min(i / (NC * 64), Q - 1) * K;
    qs[i / (NC * 64)][i % (NC * 64)] =
        at < K ? *reinterpret_cast<const f32x4*>(from + at)
               : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  __syncthreads();
  const int b = blockIdx.x, G = gridDim.x;
  const int g0 = (int)((long)N * b / G), g1 = (int)((long)N * (b + 1) / G);
  const int r0 = g0 + (g1 - g0) * wid / SF_WAVES;
  const int r1 = g0 + (g1 - g0) * (wid + 1) / SF_WAVES;
  // this wave's best so far, lane i the i-th: number of float32's order, row
  unsigned int best[QN], least[QN];  // least: the k-th
  int row[QN];
  float own[QN];  // of this lane's row of the 64 at hand
#pragma unroll
  for (int j = 0; j < QN; ++j) {
    best[j] = least[j] = 0;
    row[j] = -1;
    own[j] = 0.f;
  }
  const bool in = (NC - 1) * 256 + lane * 4 < K;
  for (int s0 = r0; s0 < r1; s0 += 64) {
    const int s1 = min(s0 + 64, r1);
    for (int r = s0; r < s1; r += 4) {
      f32x4 x[4][NC];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float* from = corpus + (long)min(r + i, s1 - 1) * K + lane * 4;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          x[i][c] = {0.f, 0.f, 0.f, 0.f};
          if (c < NC - 1 || in)
            x[i][c] = *reinterpret_cast<const f32x4*>(from + c * 256);
        }
      }
      float s[QN][4];
#pragma unroll
      for (int j = 0; j < QN; ++j) {
#pragma unroll
        for (int i = 0; i < 4; ++i) s[j][i] = 0.f;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const f32x4 y = qs[j][c * 64 + lane];
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              s[j][i] = fmaf(x[i][c][e], y[e], s[j][i]);
        }
      }
#pragma unroll
      for (int j = 0; j < QN; ++j) {
        const int sum = __builtin_bit_cast(int, sf_sums(s[j]));
        int to = __builtin_bit_cast(int, own[j]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int v = __builtin_amdgcn_readlane(sum, (i * 2 & 3) * 16 +
                                                           (i >> 1) * 16);
          to = lane == r - s0 + i ? v : to;
        }
        own[j] = __builtin_bit_cast(float, to);
      }
    }
    const int n = s1 - s0;
#pragma unroll
    for (int j = 0; j < QN; ++j) {
      const unsigned int u = f32_to_ord(own[j]);
      if (s0 == r0) {
        int rank = 0;
        for (int i = 0; i < n; ++i) {
          const unsigned int o = __builtin_amdgcn_readlane(u, i);
          rank += o > u || (o == u && i < lane);
        }
        if (lane >= n) rank = lane;  // those that are, take 0 to n - 1
        best[j] = __builtin_amdgcn_ds_permute(rank * 4, lane < n ? (int)u : 0);
        row[j] = __builtin_amdgcn_ds_permute(rank * 4, lane < n ? s0 + lane : -1);
        least[j] = __builtin_amdgcn_readlane(best[j], k - 1);
      } else {
        // (64 rows, more than k, are behind these)
        unsigned long long some = __ballot(lane < n && u > least[j]);
        while (some) {
          const int i = __ffsll(some) - 1;
          some &= some - 1;
          const unsigned int w = __builtin_amdgcn_readlane(u, i);
          const int at = __popcll(__ballot(row[j] >= 0 && best[j] >= w));
          const unsigned int v = __shfl_up(best[j], 1, 64);
          const int o = __shfl_up(row[j], 1, 64);
          best[j] = lane < at ? best[j] : lane == at ? w : v;
          row[j] = lane < at ? row[j] : lane == at ? s0 + i : o;
        }
        least[j] = __builtin_amdgcn_readlane(best[j], k - 1);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < QN; ++j)
    // 0 where there is none: a row's key is not, for its place
    if (lane < k)
      key[j][wid][lane] =
          ((unsigned long long)best[j] << 32) | (unsigned int)~row[j];
  if (tid < QN) count[tid] = 0;
  __syncthreads();
  // the k-th largest of the waves' first four bounds the k-th largest of all
  // from below; what reaches it is ranked
  if (wid < Q) {
    unsigned int u = 0;
    if ((lane & 3) < k) u = (unsigned int)(key[wid][lane >> 2][lane & 3] >> 32);
    int rank = 0;
#pragma unroll 8
    for (int i = 0; i < 64; ++i) {
      const unsigned int o = __builtin_amdgcn_readlane(u, i);
      rank += o > u || (o == u && i < lane);
    }
    if (rank == k - 1) bound[wid] = u;
  }
  __syncthreads();
  for (int i = tid; i < Q * SF_WAVES * k; i += SF_WAVES * 64) {
    const int j = i / (SF_WAVES * k), w = i / k % SF_WAVES;
    const unsigned long long mine = key[j][w][i % k];
    if (mine != 0 && (unsigned int)(mine >> 32) >= bound[j])
      some[j][atomicAdd(&count[j], 1)] = mine;
  }
  __syncthreads();
  constexpr int EACH = SF_WAVES * 64 / QN;  // threads of a query
  const int j = tid / EACH;
  if (j >= Q) return;
  const int n = count[j];
  for (int i = tid % EACH; i < n; i += EACH) {
    const unsigned long long mine = some[j][i];
    int rank = 0;
#pragma unroll 4
    for (int e = 0; e < n; ++e) rank += some[j][e] > mine;
    if (rank < k) {
      const long at = ((long)j * G + b) * (k | 1) + rank;
      out_v[at] = ord_to_f32((unsigned int)(mine >> 32));
      out_i[at] = (int)~(unsigned int)mine;
    }
  }
  if (k % 2 == 0 && tid % EACH == 0) {
    const long at = ((long)j * G + b) * (k | 1) + k;
    out_v[at] = ord_to_f32(0);
    out_i[at] = -1;
  }
}

// Workgroups for N >= 64 rows: each has 64 or more, so k of its own.
extern "C" int search_few_groups(int N) { return N / 64 < 256 ? N / 64 : 256; }

// Q up to 4 (K beyond 768: 2), k up to 30, K a multiple of 4 up to 1024.
extern "C" void launch_search_few(const float* q, const float* corpus,
                                  float* out_v, int* out_i, int Q, int N,
                                  int K, int k, hipStream_t stream) {
#define SF(NC, QN)                                                          \
  hipLaunchKernelGGL((search_few_kernel<NC, QN>),                           \
                     dim3(search_few_groups(N)), dim3(SF_WAVES * 64), 0,    \
                     stream, q, corpus, out_v, out_i, Q, N, K, k)
#define SF_Q(NC)            \
  do {                      \
    if (Q == 1) SF(NC, 1);  \
    else if (Q == 2) SF(NC, 2); \
    else SF(NC, 4);         \
  } while (0)
  switch ((K + 255) / 256) {
    case 1: SF_Q(1); break;
    case 2: SF_Q(2); break;
    case 3: SF_Q(3); break;
    default:
      if (Q == 1) SF(4, 1);
      else SF(4, 2);
  }
#undef SF_Q
#undef SF
}

// The k best rows of a corpus for each query, from the largest score of every four
// rows (`most`, [Q, groups] numbers of float32's order, 0 for none): the k groups
// of the largest hold the k best rows. Their rows are scored again, in plain
// float32, so the groups' numbers need only be near: a row that is left out for a
// group's is within their error of it. Equals go by place, groups as rows. A
// workgroup per query; k <= 60.
// lost and again, null where the groups' numbers have float32's error: lost[q] is what
// those of query q may be off beyond that (score_scale_kernel). Where it is more than
// 2^-22 of the k-th largest, again[q] is set to 1, and the groups made again and chosen
// from by a second launch (`second`: of such queries only).
// The k-th largest of 64 sixteens of threads bounds the k-th largest group from
// below, as in topk_regs_kernel; likewise, more than the buffer holds are selected
// byte by byte.
#define ST_THREADS 1024
#define ST_CAP 1024
// The groups are read by loops, a second time by the few threads that have some of
// the largest: written out for groups in registers the code takes longer to arrive
// than the groups (64 a thread 41 us, 16 13).
__global__ void __launch_bounds__(ST_THREADS)
search_top_kernel(const unsigned int* __restrict__ most,
                  const float* __restrict__ q,
                  const float* __restrict__ corpus, float* __restrict__ out_v,
                  int* __restrict__ out_i, int N, int groups, int K, int k,
                  const float* __restrict__ lost, int* __restrict__ again,
                  bool second) {
  __shared__ unsigned int top[16][64], hist[256], thresh, ncand, found, above,
      counts[16];
  __shared__ unsigned long long key[ST_CAP];
  __shared__ int chosen[64];
  __shared__ unsigned long long rows[256];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  if (second && again[blockIdx.x] == 0) return;
  const unsigned int* row = most + (long)blockIdx.x * groups;

  // f(number, place) for all groups of this thread
  auto each = [&](auto f) {
#pragma unroll 4
    for (int i = tid; i < groups / 4; i += ST_THREADS) {
      const i32x4 v = reinterpret_cast<const i32x4*>(row)[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) f((unsigned int)v[e], i * 4 + e);
    }
  };
  unsigned int mine = 0;
  each([&](unsigned int u, int) { mine = max(mine, u); });
  top[wid][lane] = mine;
  if (tid == 0) ncand = 0;
  __syncthreads();
  if (tid < 64) {
    unsigned int m = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) m = max(m, top[w][lane]);
    int rank = 0;
#pragma unroll
    for (int j = 0; j < 64; ++j) {
      const unsigned int o = __builtin_amdgcn_readlane(m, j);
      rank += o > m || (o == m && j < lane);
    }
    if (rank == k - 1) thresh = m;
  }
  __syncthreads();
  auto gather = [&](unsigned int from) {
    if (mine >= from && mine != 0)
      each([&](unsigned int u, int i) {
        if (u >= from && u != 0) {
          const unsigned int slot = atomicAdd(&ncand, 1u);
          if (slot < ST_CAP)
            key[slot] = ((unsigned long long)u << 32) | (unsigned int)~i;
        }
      });
    __syncthreads();
  };
  gather(thresh);
  if (ncand > ST_CAP) {
    unsigned int want = k, T = 0;
    for (int shift = 24; shift >= 0; shift -= 8) {
      if (tid < 256) hist[tid] = 0;
      __syncthreads();
      each([&](unsigned int u, int) {
        if (u != 0 && (shift == 24 || (u >> (shift + 8)) == (T >> (shift + 8))))
          atomicAdd(&hist[(u >> shift) & 255u], 1u);
      });
      __syncthreads();
      if (tid == 0) {
        unsigned int sum = 0;
        int b = 255;
        for (; b > 0 && sum + hist[b] < want; --b) sum += hist[b];
        found = b;
        above = sum;
      }
      __syncthreads();
      T |= found << shift;
      want -= above;
    }
    if (tid == 0) ncand = 0;
    __syncthreads();
    if (T != 0xffffffffu) gather(T + 1);
    // and the first `want` that equal it, a thousand places after the other
    const unsigned int first = ncand;
    unsigned int have = 0;
    for (int i0 = 0; i0 < groups && have < want; i0 += ST_THREADS) {
      const int i = i0 + tid;
      const bool equal = i < groups && row[i] == T;
      const unsigned long long m = __ballot(equal);
      if (lane == 0) counts[wid] = __popcll(m);
      __syncthreads();
      unsigned int at = have + __popcll(m & ((1ull << lane) - 1)), all = 0;
      for (int w = 0; w < 16; ++w) {
        if (w < wid) at += counts[w];
        all += counts[w];
      }
      if (equal && at < want)
        key[first + at] = ((unsigned long long)T << 32) | (unsigned int)~i;
      have += all;
      __syncthreads();
    }
    if (tid == 0) ncand = first + min(have, want);
    __syncthreads();
  }
  const int n = (int)min(ncand, (unsigned int)ST_CAP), take = min(n, k);
  if (tid < n) {
    const unsigned long long own = key[tid];
    int r = 0;
#pragma unroll 8
    for (int j = 0; j < n; ++j) r += key[j] > own;
    if (r < take) chosen[r] = (int)~(unsigned int)own;
    // (fewer groups than k have all rows)
    if (r == k - 1 && lost != nullptr && !second &&
        !(lost[blockIdx.x] <=
          0x1p-22f * fabsf(ord_to_f32((unsigned int)(own >> 32)))))
      again[blockIdx.x] = 1;
  }
  __syncthreads();
  const float* query = q + (long)blockIdx.x * K;
  for (int c = wid; c < take; c += 16) {
    const int r0 = chosen[c] * 4;
    float s[4];
    search_dot(query, corpus, r0, N, K, s);
    if (lane < 4) {
      const float v = lane == 0 ? s[0] : lane == 1 ? s[1] : lane == 2 ? s[2]
                                                                      : s[3];
      rows[c * 4 + lane] =
          r0 + lane < N ? ((unsigned long long)f32_to_ord(v) << 32) |
                              (unsigned int)~(r0 + lane)
                        : 0ull;
    }
  }
  __syncthreads();
  float* ov = out_v + (long)blockIdx.x * k;
  int* oi = out_i + (long)blockIdx.x * k;
  if (tid >= 256) return;
  const unsigned long long own = tid < take * 4 ? rows[tid] : 0ull;
  int r = 0, real = 0;
#pragma unroll 8
  for (int j = 0; j < take * 4; ++j) {
    const unsigned long long other = rows[j];
    r += other > own;
    real += other != 0;
  }
  if (own != 0 && r < k) {
    ov[r] = ord_to_f32((unsigned int)(own >> 32));
    oi[r] = (int)~(unsigned int)own;
  }
  if (tid >= real && tid < k) {
    ov[tid] = -INFINITY;
    oi[tid] = -1;
  }
}

// most: [Q, groups], groups % 4 == 0; K % 4 == 0, operands at multiples of 16 bytes
extern "C" void launch_search_top(const unsigned int* most, const float* q,
                                  const float* corpus, float* out_v,
                                  int* out_i, int Q, int N, int groups, int K,
                                  int k, const float* lost, int* again,
                                  bool second, hipStream_t stream) {
  hipLaunchKernelGGL(search_top_kernel, dim3(Q), dim3(ST_THREADS), 0, stream,
                     most, q, corpus, out_v, out_i, N, groups, K, k, lost, again,
                     second);
}

extern "C" void launch_topk_chunk(const float* scores, const int* in_idx,
                                  float* out_v, int* out_i, int Qn, long N,
                                  int chunk, int k, bool regs,
                                  hipStream_t stream) {
  const int nchunks = (int)((N + chunk - 1) / chunk);
  dim3 grid(nchunks, Qn);
  if (regs) {  // chunk <= TR_CHUNK, k <= 256
    hipLaunchKernelGGL(topk_regs_kernel, grid, dim3(256), 0, stream, scores,
                       in_idx, out_v, out_i, N, chunk, k, nchunks);
    return;
  }
  hipLaunchKernelGGL(topk_chunk_kernel, grid, dim3(256), 0, stream, scores,
                     in_idx, out_v, out_i, N, chunk, k, nchunks);
}

// ---- Hamming distance scoring (ubinary precision path) -----------------
// codes are WORD-MAJOR: codes_t [W, N] u64 (W = nbits/64) so candidate
// reads coalesce; query: [Q, W] u64. out: [Q, N] f32 = -hamming.
__global__ void __launch_bounds__(256)
hamming_score_kernel(const unsigned long long* __restrict__ qcodes,
                     const unsigned long long* __restrict__ codes_t,
                     float* __restrict__ out, long N, int W) {
  const int q = blockIdx.y;
  const long stride = (long)gridDim.x * blockDim.x;
  // query words via L2/L1 (small)
  for (long n = (long)blockIdx.x * blockDim.x + threadIdx.x; n < N;
       n += stride) {
    int d = 0;
    for (int w = 0; w < W; ++w)
      d += __popcll(qcodes[(long)q * W + w] ^ codes_t[(long)w * N + n]);
    out[(long)q * N + n] = -(float)d;
  }
}

extern "C" void launch_hamming_score(const void* qcodes, const void* codes_t,
                                     float* out, int Qn, long N, int W,
                                     hipStream_t stream) {
  int bl = (int)min((N + 255) / 256, (long)2048);
  dim3 grid(bl, Qn);
  hipLaunchKernelGGL(hamming_score_kernel, grid, dim3(256), 0, stream,
                     (const unsigned long long*)qcodes,
                     (const unsigned long long*)codes_t, out, N, W);
}

// ---- batched IVF chunk scoring (approximate search) --------------------
// slabs: [nchunks, cap, H] f32 padded chunk slabs; probes: [Q*nprobe]
// int32 chunk ids; qv: [Q, H] f32; out: [Q*nprobe*cap] f32 (-inf at
// pad rows). One block per (query, probe): the query vector is staged
// in LDS once; each wave streams rows of the contiguous slab with
// 16-byte-per-lane coalesced loads and a wave-reduce dot. BW-bound by
// design (bf16 slabs read once; winners re-scored fp32 host-side).
__global__ void __launch_bounds__(256)
ivf_score_kernel(const float* __restrict__ slabs,
                 const int* __restrict__ lens,
                 const int* __restrict__ probes,
                 const float* __restrict__ qv, float* __restrict__ out,
                 int nprobe, int cap, int H) {
  extern __shared__ __attribute__((aligned(16))) float qlds[];
  const int qi = blockIdx.x / nprobe;
  const int ch = probes[blockIdx.x];
  const int len = lens[ch];
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;

  for (int i = threadIdx.x; i < H; i += 256) qlds[i] = qv[qi * H + i];
  __syncthreads();

  const float* slab = slabs + (long)ch * cap * H;
  float* orow = out + (long)blockIdx.x * cap;
  const int span = 64 * 4;  // elements covered per wave pass
  for (int r = wid; r < cap; r += 4) {
    float acc = 0.f;
    if (r < len) {
      const float* row = slab + (long)r * H;
      for (int i0 = lane * 4; i0 < H; i0 += span) {
        // 4 f32 = one 16-byte load (tail guard per element)
        if (i0 + 4 <= H) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(row + i0);
#pragma unroll
          for (int j = 0; j < 4; ++j) acc += v[j] * qlds[i0 + j];
        } else {
          for (int j = i0; j < H; ++j) acc += row[j] * qlds[j];
        }
      }
      acc = wave_reduce_sum(acc);
    }
    if (lane == 0) orow[r] = (r < len) ? acc : -INFINITY;
  }
}

extern "C" void launch_ivf_score(const void* slabs, const int* lens,
                                 const int* probes, const float* qv,
                                 float* out, int nblocks, int nprobe,
                                 int cap, int H, hipStream_t stream) {
  hipLaunchKernelGGL(ivf_score_kernel, dim3(nblocks), dim3(256),
                     H * (int)sizeof(float), stream,
                     (const float*)slabs, lens, probes, qv, out,
                     nprobe, cap, H);
}
