// kNN search kernels replacing faiss-gpu (reference rag/search.py:231-399):
// chunked radix-select top-k over a score matrix,
// and packed-binary Hamming scoring for the ubinary precision path.
//
// Pipeline (python side, rag/search.py here):
//   scores_chunk = Q @ C_chunk^T          (hipBLASLt or gemm.hip)
//   topk_chunk_kernel -> per-chunk candidates
//   topk over concatenated candidates (same kernel, with idx indirection)
//
// topk_regs_kernel takes small k (the caller's choice); beyond,
// topk_chunk_kernel: one 256-thread block per (query, chunk). Two-round
// 8-bit radix select over monotonic uint32 keys finds a threshold, a
// compact pass gathers candidates (cap 2048) into LDS, a bitonic sort
// orders them, and the top k (vals + indices) are written out.
#include "common.h"

#define TK_CAP 2048  // candidate buffer (vals+idx) in LDS

__device__ __forceinline__ unsigned int f32_to_ord(float f) {
  union { float f; unsigned int u; } c;
  c.f = f;
  return (c.u & 0x80000000u) ? ~c.u : (c.u | 0x80000000u);
}
__device__ __forceinline__ float ord_to_f32(unsigned int u) {
  union { float f; unsigned int u; } c;
  c.u = (u & 0x80000000u) ? (u & 0x7fffffffu) : ~u;
  return c.f;
}

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
