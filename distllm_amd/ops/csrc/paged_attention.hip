// Paged-KV decode attention (single new token per sequence).
// Replaces vLLM's paged attention (reference delegated generation to
// vLLM, generate/generators/vllm_backend.py).
//
// Cache layout: kcache/vcache [nblocks, HKV, BLK, D], BLK=16, bf16 or OCP
// fp8 e4m3 (CDNA4-native; halves decode KV bandwidth, doubles capacity;
// values are stored unscaled, |k|,|v| << 448 in practice).
// block_table [B, max_blocks] int32 ; ctx_len [B] int32.
// q: [B, H, D] bf16, rows of any stride ; out: [B, H, D] bf16.
//
// Bound by reading the cache. A workgroup has the query heads of one key
// head (up to 16 of them: the columns of the products) and a share of the
// sequence; its 4 waves take tiles of 32 keys (two pages) in turn and work
// alone until their softmax states meet in LDS.
//  - bf16 pages go to the wave's own ring of LDS buffers as they lie in the
//    cache, whole lines by global_load_lds; fp8 pages pass through registers,
//    the next tile's loads in flight, and are widened on the way.
//  - scores are mfma(K, Q^T), keys on rows and heads on lanes, the output is
//    mfma(V^T, P), columns on rows and heads on lanes, V transposed on its
//    way out of LDS. Softmax state and rescaling are lane-local but for the
//    maximum over the four groups of lanes that share a head.
//  - probabilities stay fp32: each goes in as the sum of three bf16 numbers,
//    which is exactly it (two leave 2^-17 of it, and what two values that
//    cancel leave can be less than that). With bf16 pages no part is negative
//    or, but for a first one, 0: an infinite value gives an infinite result. fp8
//    has no infinities.
//  - NS workgroups share a sequence where B * HKV is small; a second launch
//    joins them or, in a decode step, the last of them.
//  - a decode step goes by the STEP form alone (launch_step_attn). launch_paged_attn
//    and launch_rope_put are what ops.paged_attn and ops.rope_put have for callers
//    that attend by themselves; no model of this package does.
//  - a decode step's queries are rotated and its key and value put into the
//    cache in the same launch (STEP): us in a graph, three launches and one,
//    32 heads on 8, B = 1, 2048 tokens 12.7 -> 7.6, 64 tokens 10.9 -> 6.3, B = 8
//    of 500 11.0 -> 7.4, B = 64 of 200 to 2027 70 -> 56, and 51 with the sequences
//    cut and ordered by their lengths (step_plan_kernel).
// Measured, us, with kernels that read a key row per lane and a value element
// per lane, and now (32 heads on 8 of 128, bf16; fp8): B = 1, 2048 cached
// tokens 32 -> 11.0 (31 -> 11.1); B = 16 of 100 to 4000 115 -> 36.5 (104 ->
// 24); B = 64 of 200 to 2048 137 -> 61, 4.8 TB/s (117 -> 38); B = 128 of 1000
// 150 -> 98, 5.3 TB/s (96 -> 56). With copies that the compiler knows of, which
// the reads of V then wait for, also for the next tile's: 39, 65 and 101.
// Those kernels are still the faster ones where contexts of a page or two meet
// 16 key heads and rows or more (64 x 32 heads of 128, of 16: 11, now 19): which
// kernel runs is the host's choice, and the lengths are on the device only (where
// step_plan_kernel deals a step's shares by them).
#include "ahead.h"
#include "common.h"
#include <hip/hip_fp8.h>

#define PBLK 16  // tokens per KV block
#define KT 32    // keys of a tile

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

extern __shared__ __attribute__((aligned(16))) char smem[];

union pa_frag {
  bf16x8 v;
  s16x4 h[2];
  unsigned int d[4];
};

__device__ __forceinline__ unsigned int pa_pack(float a, float b) {
  return __builtin_bit_cast(
      unsigned int, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

// 16 fp8 numbers as 16 bf16 (exact)
__device__ __forceinline__ void pa_widen(const i32x4 v, i32x4 (&out)[2]) {
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8(v[w], false);
    const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8(v[w], true);
    out[w >> 1][(w & 1) * 2] = (int)pa_pack(lo[0], lo[1]);
    out[w >> 1][(w & 1) * 2 + 1] = (int)pa_pack(hi[0], hi[1]);
  }
}

// Cache element of a bf16 number.
__device__ __forceinline__ void cache_store(unsigned short* p,
                                            unsigned short v) {
  *p = v;
}
__device__ __forceinline__ void cache_store(unsigned char* p,
                                            unsigned short v) {
  *p = __hip_fp8_e4m3(bf2f(v)).__x;
}

// A decode step's projections [B, H + 2 HKV, D], as bf16 numbers or, S > 0, as
// the S fp32 slabs of a product whose K was shared, without its bias; rotation
// tables [positions, D / 2].
struct PaStep {
  const unsigned short* qkv;
  const float* parts;
  int S;
  const unsigned short* bias;
  const float *cs, *sn;
  // the launch's shares (step_plan_kernel), eight numbers each: sequence or -1,
  // its length, first tile, the one behind the last; of the sequence, the first
  // share and their number. The seventh of the first B is not a share's but that
  // row's: whether another row of the step is an earlier token of its sequence
  const int* slots;
  Ahead ahead;
};

// Columns c .. c + 3 and D / 2 + c .. of head h of row b, as bf16 numbers; ROT:
// rotated (half-split, fp32) by the angles of position pos.
template <int D>
__device__ __forceinline__ void step_columns(const PaStep& p, int B,
                                             int heads, int b, int h, int c,
                                             bool rotate, int pos,
                                             unsigned short* a,
                                             unsigned short* e) {
  const long at = ((long)b * heads + h) * D + c;
  f32x4 co = {1.f, 1.f, 1.f, 1.f}, si = {0.f, 0.f, 0.f, 0.f};
  if (rotate) {
    co = *reinterpret_cast<const f32x4*>(p.cs + (long)pos * (D / 2) + c);
    si = *reinterpret_cast<const f32x4*>(p.sn + (long)pos * (D / 2) + c);
  }
  if (p.S == 0) {
    *reinterpret_cast<i32x2*>(a) = *reinterpret_cast<const i32x2*>(p.qkv + at);
    *reinterpret_cast<i32x2*>(e) =
        *reinterpret_cast<const i32x2*>(p.qkv + at + D / 2);
  } else {
    f32x4 va = {0.f, 0.f, 0.f, 0.f}, ve = va;
    const long slab = (long)B * heads * D;
    // four slabs at once are on their way
    for (int s0 = 0; s0 < p.S; s0 += 4) {
      f32x4 pa[4], pe[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const float* from = p.parts + min(s0 + s, p.S - 1) * slab + at;
        pa[s] = *reinterpret_cast<const f32x4*>(from);
        pe[s] = *reinterpret_cast<const f32x4*>(from + D / 2);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          va[j] = s0 + s < p.S ? va[j] + pa[s][j] : va[j];
          ve[j] = s0 + s < p.S ? ve[j] + pe[s][j] : ve[j];
        }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (p.bias != nullptr) {
        va[j] += bf2f(p.bias[h * D + c + j]);
        ve[j] += bf2f(p.bias[h * D + D / 2 + c + j]);
      }
      a[j] = f2bf(va[j]);
      e[j] = f2bf(ve[j]);
    }
  }
  if (rotate) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float x = bf2f(a[j]), y = bf2f(e[j]);
      // fused as written, in every kernel alike
      a[j] = f2bf(fmaf(x, co[j], -(y * si[j])));
      e[j] = f2bf(fmaf(y, co[j], x * si[j]));
    }
  }
}

// Two results of a workgroup for the kernel, or (JOIN) the workgroup, that joins
// them.
template <bool JOIN>
__device__ __forceinline__ void pa_put(float* to, float a, float b) {
  const f32x2 v = {a, b};
  if constexpr (JOIN)
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(to),
                       __builtin_bit_cast(unsigned long long, v),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else
    *reinterpret_cast<f32x2*>(to) = v;
}
__device__ __forceinline__ f32x2 pa_get(const float* from) {
  return __builtin_bit_cast(
      f32x2, __hip_atomic_load(
                 reinterpret_cast<const unsigned long long*>(from),
                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// LDS of a workgroup: the waves' rings of R tiles of K and V, then their states
constexpr int NW = 4;  // waves of a workgroup
constexpr int pa_lds(int D, int R) {
  const int ring = NW * R * 2 * KT * D * 2, states = NW * 16 * (D + 2) * 4;
  return ring > states ? ring : states;
}

// The attention of a few sequences is latency and leaves the memory idle. The
// last workgroups of its launch read the weights of the product behind it
// meanwhile, each run of 16 rows into the L2 of the XCD on which the product's
// workgroup will be (they go round), and so into the cache that all share. A CU
// takes in some 50 GB/s this way, so it wants most of them: us of a step of 8
// layers, one sequence of 2048, 32 workgroups 928, 64 840, 128 801, 192 803, none
// 821; of 32 tokens 925, 832, 786, 760 and 778; 8 of 100 1005, 912, 850, 840, 867;
// 8-bit weights, 2048 606, 572, 576, 571, 578. (The same behind norms of 5 us
// shortened the products by less than it lengthened the norms.)
__device__ __forceinline__ void fetch_ahead(const Ahead& a) {
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int xcd = blockIdx.x % 8, waves = a.blocks / 8 * NW;
  const int turn = (blockIdx.x - (gridDim.x - a.blocks)) / 8;
  const int n = (a.chunks - xcd + 7) / 8 * a.pieces;
  int k = 0;
  for (int i = turn * NW + wid; i < n; i += waves) {
    const long piece =
        (xcd + (long)(i / a.pieces) * 8) * a.pieces + i % a.pieces;
    // all to one place in LDS, where nobody looks: through registers, eight at a
    // time, a step of one sequence of 2048 took 836
    copy_to_lds(a.from + piece * 1024 + lane * 16, smem + wid * 1024);
    if ((++k & 7) == 0) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// ALIGNED: the pages start at a multiple of 16 bytes, as the copies to LDS ask;
// else bf16 pages pass through registers like fp8 ones, one tile after another.
// STEP: queries come out of the step's projections and are rotated here, into
// LDS, while the first tile is on its way, and so are the new token's key and
// value where the share ends with it: the wave that has the last tile puts them
// into it, and they go to the cache (from the first of several groups of heads).
// A launch that did this ahead (rope_put_kernel) took 4.7 us.
// Rows of one step may be tokens of one sequence that follow each other. Nothing
// orders this launch's workgroups, so those of a later token put the earlier ones
// into the cache themselves, too, with the same numbers, ahead of their first tile.
template <int D, bool FP8, bool ALIGNED, int R, bool STEP>
__global__ void __launch_bounds__(256)
paged_attn_kernel(const unsigned short* __restrict__ q, long q_stride,
                  const PaStep step, char* kcache, char* vcache,
                  const int* __restrict__ block_table,
                  const int* __restrict__ ctx_len,
                  unsigned short* __restrict__ out,
                  float* pacc, float* pml, int* arrived, int B, int H, int HKV,
                  int max_blocks, int NS, float scale) {
  constexpr int NCH = D / 8;            // 16-byte pieces of a bf16 row
  constexpr int ROWS = 1024 / (2 * D);  // rows of a 1 KiB piece of a tile
  constexpr int PIECES = KT / ROWS;     // pieces of K or V of a tile
  constexpr int TILE = KT * D * 2;      // bytes of K or V of a tile
  constexpr int DB = D / 16;
  if constexpr (STEP) {
    if (blockIdx.x >= gridDim.x - step.ahead.blocks) {
      // where there are more pages than weights to read, the time is theirs: us
      // of a step of 8 sequences of 2048 990 without, 995 with
      long cached = 0;
      for (int i = 0; i < B; ++i) cached += ctx_len[i];
      if (cached * HKV * D * (FP8 ? 2 : 4) <=
          (long)step.ahead.chunks * step.ahead.pieces * 1024)
        fetch_ahead(step.ahead);
      return;
    }
  }
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, g = lane >> 4;
  const int GR = H / HKV, NG = (GR + 15) / 16;
  const int slot = STEP ? blockIdx.x / (NG * HKV) : 0;
  const int split = STEP ? 0 : blockIdx.x % NS;
  const int hg = STEP ? blockIdx.x % NG : blockIdx.x / NS % NG;
  const int kvh = STEP ? blockIdx.x / NG % HKV : blockIdx.x / NS / NG % HKV;
  int share[6] = {};
  if constexpr (STEP) {
#pragma unroll
    for (int i = 0; i < 6; ++i)
      share[i] = __builtin_amdgcn_readfirstlane(step.slots[slot * 8 + i]);
    if ((unsigned)share[0] >= (unsigned)B) return;
    NS = share[5];
  }
  const int b = STEP ? share[0] : blockIdx.x / NS / NG / HKV;
  const int head0 = kvh * GR + hg * 16, nh = min(GR - hg * 16, 16);

  const int ctx = STEP ? share[1] : ctx_len[b];
  const int L = min(ctx, max_blocks * PBLK);
  const int T = (L + KT - 1) / KT, per = (T + NS - 1) / NS;
  const int first_tile = STEP ? share[2] : split * per;
  const int t0 = first_tile + wid;
  const int t1 = STEP ? share[3] : min(T, split * per + per);
  const int mine = t1 > t0 ? (t1 - t0 + NW - 1) / NW : 0;  // t0, t0 + NW, ...
  const int last_page = max(L - 1, 0) / PBLK;
  const int* bt = block_table + (long)b * max_blocks;
  const long page_bytes = (long)HKV * PBLK * D * (FP8 ? 1 : 2);
  const long head_bytes = (long)kvh * PBLK * D * (FP8 ? 1 : 2);

  // page numbers of the wave's next 32 tiles, two a tile, on the lanes
  int pages = 0;
  auto fetch_pages = [&](int i) {
    const int p = (t0 + (i + (lane >> 1)) * NW) * 2 + (lane & 1);
    pages = mine > 0 ? bt[min(p, last_page)] : 0;
  };
  auto page = [&](int i, int half) {
    return __builtin_amdgcn_readlane(pages, (i & 31) * 2 + half);
  };
  char* ring = smem + wid * R * 2 * TILE;

  // bf16: pieces of K and V of tile i, pieces of 16 bytes XOR-ed with the
  // row in K, of 32 bytes in V
  auto issue = [&](int i) {
    char* dst = ring + (i % R) * 2 * TILE;
    const int r = lane / NCH, c = lane % NCH;
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      const int row = p * ROWS + r;
      const long at = page(i, p * ROWS / PBLK) * page_bytes + head_bytes +
                      (row % PBLK) * (D * 2);
      to_lds<ALIGNED>(kcache + at + ((c ^ (row & (NCH - 1))) * 16),
                      dst + p * 1024);
      to_lds<ALIGNED>(vcache + at + ((c ^ ((row & 3) << 1)) * 16),
                      dst + TILE + p * 1024);
    }
  };
  // fp8: the same rows through registers, 16 numbers a load
  constexpr int LOADS = FP8 ? KT * D / 1024 : 1;
  i32x4 kreg[LOADS], vreg[LOADS];
  auto issue8 = [&](int i) {
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      const int at = (j * 64 + lane) * 16, row = at / D, col = at % D;
      const int pg = row < PBLK ? page(i, 0) : page(i, 1);
      const long off = pg * page_bytes + head_bytes + (row % PBLK) * D + col;
      kreg[j] = *reinterpret_cast<const i32x4_any*>(kcache + off);
      vreg[j] = *reinterpret_cast<const i32x4_any*>(vcache + off);
    }
  };
  auto store8 = [&]() {
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      const int at = (j * 64 + lane) * 16, row = at / D, c = at % D / 8;
      i32x4 w[2];
      pa_widen(kreg[j], w);
#pragma unroll
      for (int e = 0; e < 2; ++e)
        *reinterpret_cast<i32x4*>(
            ring + row * (2 * D) + ((c + e) ^ (row & (NCH - 1))) * 16) = w[e];
      pa_widen(vreg[j], w);
#pragma unroll
      for (int e = 0; e < 2; ++e)
        *reinterpret_cast<i32x4*>(
            ring + TILE + row * (2 * D) + ((c + e) ^ ((row & 3) << 1)) * 16) =
            w[e];
    }
  };

  const int pos = ctx - 1, heads = H + 2 * HKV;
  // Numbers c .. and D / 2 + c .. of a row of the cache; of fp8 pages they come
  // back as what the cache then holds.
  auto put = [&](char* to, int c, unsigned short* a, unsigned short* e,
                 bool write) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      unsigned short* x = half ? e : a;
      const int col = c + half * (D / 2);
      if constexpr (FP8) {
        unsigned char eight[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          cache_store(&eight[i], x[i]);
          __hip_fp8_e4m3 f;
          f.__x = eight[i];
          x[i] = f2bf((float)f);
        }
        if (write)
#pragma unroll
          for (int i = 0; i < 4; ++i) to[col + i] = (char)eight[i];
      } else if (write) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          reinterpret_cast<unsigned short*>(to)[col + i] = x[i];
      }
    }
  };
  fetch_pages(0);
  if constexpr (STEP) {
    if (B > 1 && step.slots[b * 8 + 6] != 0) {
      for (int j = 0; j < B; ++j) {
        const int p = ctx_len[j] - 1;
        if (j == b || p < 0 || p >= pos || p / PBLK >= max_blocks) continue;
        const int pg = block_table[(long)j * max_blocks + p / PBLK];
        if (bt[p / PBLK] != pg || threadIdx.x >= D / 4) continue;
        const int row = threadIdx.x / (D / 8), c = threadIdx.x % (D / 8) * 4;
        unsigned short a[4], e[4];
        step_columns<D>(step, B, heads, j, H + row * HKV + kvh, c, row == 0, p,
                        a, e);
        put((row == 0 ? kcache : vcache) + pg * page_bytes + head_bytes +
                (long)(p % PBLK) * D * (FP8 ? 1 : 2),
            c, a, e, true);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      __syncthreads();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
  }

  // the first tile is on its way while the queries come
  int at = 0;  // tiles issued
  auto next = [&]() {
    if (at > 0 && (at & 31) == 0) fetch_pages(at);
    if constexpr (FP8) issue8(at++);
    else issue(at++);
  };
  while (at < (R > 1 ? R - 1 : 1) && at < mine) next();

  // of the workgroup, of the wave: its share ends with the new token
  const bool newest = STEP && pos >= 0 && pos < max_blocks * PBLK && T > 0 &&
                      T - 1 >= first_tile && T - 1 < t1;
  const bool renews = newest && mine > 0 && t0 + (mine - 1) * NW == T - 1;
  // rotated queries, the new key and value: rows of D in LDS
  char* rows = smem + pa_lds(D, R);
  if constexpr (STEP) {
    const int units = (nh + (newest ? 2 : 0)) * (D / 8);
    for (int u = threadIdx.x; u < units && pos >= 0; u += NW * 64) {
      const int row = u / (D / 8), c = u % (D / 8) * 4;
      const int h = row < nh ? head0 + row
                             : H + (row - nh) * HKV + kvh;
      unsigned short a[4], e[4];
      step_columns<D>(step, B, heads, b, h, c, row <= nh, pos, a, e);
      if (row >= nh)
        put((row == nh ? kcache : vcache) + bt[pos / PBLK] * page_bytes +
                head_bytes + (long)(pos % PBLK) * D * (FP8 ? 1 : 2),
            c, a, e, hg == 0);
      *reinterpret_cast<i32x2*>(rows + (row * D + c) * 2) =
          *reinterpret_cast<const i32x2*>(a);
      *reinterpret_cast<i32x2*>(rows + (row * D + c + D / 2) * 2) =
          *reinterpret_cast<const i32x2*>(e);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
  bf16x8 qf[D / 32];
#pragma unroll
  for (int s = 0; s < D / 32; ++s) {
    pa_frag f;
#pragma unroll
    for (int i = 0; i < 4; ++i) f.d[i] = 0;
    if (c16 < nh) {
      if constexpr (STEP)
        f.v = *reinterpret_cast<const bf16x8*>(
            rows + (c16 * D + s * 32 + g * 8) * 2);
      else
        f.v = *reinterpret_cast<const bf16x8*>(
            q + b * q_stride + (long)(head0 + c16) * D + s * 32 + g * 8);
    }
    qf[s] = f.v;
  }

  // the new token's row of the last tile, which holds what was in the cache
  auto renew = [&](int i) {
    const int row = (L - 1) % KT, c = lane % NCH;
    char* kt = ring + (i % R) * 2 * TILE + row * (2 * D);
    if (lane < 2 * NCH) {
      const i32x4 x = *reinterpret_cast<const i32x4*>(
          rows + (nh + lane / NCH) * (2 * D) + c * 16);
      if (lane < NCH)
        *reinterpret_cast<i32x4*>(kt + ((c ^ (row & (NCH - 1))) * 16)) = x;
      else
        *reinterpret_cast<i32x4*>(kt + TILE + ((c ^ ((row & 3) << 1)) * 16)) =
            x;
    }
    wave_sync();
  };

  const float scale2 = scale * 1.4426950408889634f;
  float m = -1e30f, l = 0.f;  // l: of the keys of this lane group
  f32x4 acc[DB];
#pragma unroll
  for (int d = 0; d < DB; ++d) acc[d] = {0.f, 0.f, 0.f, 0.f};

  auto compute = [&](int i) {
    char* kt = ring + (i % R) * 2 * TILE;
    char* vt = kt + TILE;
    const int left = L - (t0 + i * NW) * KT;  // keys of the tile, if < 32
    if (left < KT) {
      // what lies behind the last key must not meet its zero probability
      for (int k = left * (2 * D) + lane * 16; k < TILE; k += 1024)
        *reinterpret_cast<i32x4*>(vt + k) = i32x4{0, 0, 0, 0};
    }
    f32x4 sc[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      sc[kb] = {0.f, 0.f, 0.f, 0.f};
      const int key = kb * 16 + c16;
#pragma unroll
      for (int s = 0; s < D / 32; ++s) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(
            kt + key * (2 * D) + (((s * 4 + g) ^ (key & (NCH - 1))) * 16));
        sc[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[s], sc[kb], 0,
                                                         0, 0);
      }
    }
    float top = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float s =
            kb * 16 + g * 4 + r < left ? sc[kb][r] * scale2 : -INFINITY;
        sc[kb][r] = s;
        top = fmaxf(top, s);
      }
    top = lanes_max<32>(lanes_max<16>(top));
    if (!__all(top <= m)) {
      const float mn = fmaxf(m, top);
      const float alpha = __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      l *= alpha;
#pragma unroll
      for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[d][r] *= alpha;
    }
    pa_frag part[3];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 4; r += 2) {
        float p0 = __builtin_amdgcn_exp2f(sc[kb][r] - m);
        float p1 = __builtin_amdgcn_exp2f(sc[kb][r + 1] - m);
        l += p0 + p1;
#pragma unroll
        for (int e = 0; e < 3; ++e) {
          if constexpr (FP8) {  // no infinities, and rounding costs less
            const unsigned int h = pa_pack(p0, p1);
            part[e].d[kb * 2 + r / 2] = h;
            p0 -= __builtin_bit_cast(float, h << 16);
            p1 -= __builtin_bit_cast(float, h & 0xffff0000u);
          } else {
            part[e].d[kb * 2 + r / 2] = split_bf16(p0, p1);
          }
        }
      }
    // columns 16 d .. of V, keys 4 g .. 4 g + 3 of both halves: the order in
    // which a lane holds its probabilities
    const int row = g * 4 + (c16 >> 2);
#pragma unroll
    for (int d = 0; d < DB; ++d) {
      pa_frag vf;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
        vf.h[kb] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)(
                vt + (kb * 16 + row) * (2 * D) +
                ((d ^ (row & 3)) * 32) + (c16 & 3) * 8));
#pragma unroll
      for (int e = 0; e < 3; ++e)
        acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.v, part[e].v,
                                                         acc[d], 0, 0, 0);
    }
    // the buffer is read before the wave fills it again
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };

  for (int i = 0; i < mine; ++i) {
    if constexpr (FP8) {
      store8();
      if (at < mine) next();
      wave_sync();
    } else {
      if (at < mine && at < i + R) next();
      if (at == i + R)
        asm volatile("s_waitcnt vmcnt(%0)" ::"i"((R - 1) * 2 * PIECES)
                     : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if constexpr (!ALIGNED) wave_sync();
    }
    if (renews && i == mine - 1) renew(i);
    compute(i);
  }

  // ---- the waves' states meet ---------------------------------------------
  l = lanes_sum<32>(lanes_sum<16>(l));
  __syncthreads();
  float* ml = reinterpret_cast<float*>(smem);  // [NW][16][2]
  float* wacc = ml + NW * 16 * 2;              // [NW][16][D]
  if (g == 0) {
    ml[(wid * 16 + c16) * 2] = m;
    ml[(wid * 16 + c16) * 2 + 1] = l;
  }
#pragma unroll
  for (int d = 0; d < DB; ++d)
    *reinterpret_cast<f32x4*>(wacc + (wid * 16 + c16) * D + d * 16 + g * 4) =
        acc[d];
  __syncthreads();
  // row of the share's first head among the partial results
  const long part = STEP ? (long)slot * H + head0
                         : ((long)(b * HKV + kvh) * NS + split) * GR + hg * 16;
  for (int i = threadIdx.x; i < nh * (D / 4); i += NW * 64) {
    const int head = i / (D / 4), col = i % (D / 4) * 4;
    float M = -1e30f;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, ml[(w * 16 + head) * 2]);
    float sum = 0.f;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float a = __builtin_amdgcn_exp2f(ml[(w * 16 + head) * 2] - M);
      sum += ml[(w * 16 + head) * 2 + 1] * a;
      const f32x4 v =
          *reinterpret_cast<const f32x4*>(wacc + (w * 16 + head) * D + col);
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] += a * v[r];
    }
    if (NS == 1) {
      const float inv = sum > 0.f ? 1.f / sum : 0.f;
      const i32x2 two = {(int)pa_pack(o[0] * inv, o[1] * inv),
                         (int)pa_pack(o[2] * inv, o[3] * inv)};
      *reinterpret_cast<i32x2*>(out + ((long)b * H + head0 + head) * D + col) =
          two;
    } else {
      float* to = pacc + (part + head) * D + col;
      pa_put<STEP>(to, o[0], o[1]);
      pa_put<STEP>(to + 2, o[2], o[3]);
      if (col == 0) pa_put<STEP>(pml + (part + head) * 2, M, sum);
    }
  }
  if constexpr (STEP) {
    // The last of a sequence's workgroups joins their results, which saves a
    // launch (4.7 us). Results and count are agent-scope atomics, which meet in
    // memory that all XCDs see; every wave's are there before the barrier ahead of
    // the count.
    if (NS == 1) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int* last = reinterpret_cast<int*>(smem);
    if (threadIdx.x == 0)
      *last = __hip_atomic_fetch_add(arrived + (b * HKV + kvh) * NG + hg, 1,
                                     __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT) == NS - 1;
    __syncthreads();
    if (!*last) return;
    const long first = (long)share[4] * H + head0;
    float* state = reinterpret_cast<float*>(smem) + 4;  // [NS][nh][2]
    for (int i = threadIdx.x; i < NS * nh; i += NW * 64)
      *reinterpret_cast<f32x2*>(state + i * 2) =
          pa_get(pml + (first + (long)(i / nh) * H + i % nh) * 2);
    __syncthreads();
    for (int i = threadIdx.x; i < nh * (D / 2); i += NW * 64) {
      const int head = i / (D / 2), col = i % (D / 2) * 2;
      const float* from = pacc + (first + head) * D + col;
      const float* st = state + head * 2;
      float M = -1e30f, sum = 0.f;
      for (int s = 0; s < NS; ++s) M = fmaxf(M, st[s * nh * 2]);
      f32x2 o = {0.f, 0.f};
#pragma unroll 8
      for (int s = 0; s < NS; ++s) {
        const float a = __builtin_amdgcn_exp2f(st[s * nh * 2] - M);
        const f32x2 v = pa_get(from + (long)s * H * D);
        sum += a * st[s * nh * 2 + 1];
        o[0] += a * v[0];
        o[1] += a * v[1];
      }
      const float inv = sum > 0.f ? 1.f / sum : 0.f;
      *reinterpret_cast<unsigned int*>(out + ((long)b * H + head0 + head) * D +
                                       col) = pa_pack(o[0] * inv, o[1] * inv);
    }
  }
}

// Join NS partial results; a wave per (sequence, head), the shares' states on
// its lanes. NS <= 64.
template <int D>
__global__ void __launch_bounds__(256)
paged_attn_combine_kernel(const float* __restrict__ pacc,
                          const float* __restrict__ pml,
                          unsigned short* __restrict__ out, int rows, int H,
                          int HKV, int NS) {
  constexpr int DPL = D / 64;
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);  // b * H + head
  if (row >= rows) return;
  const int GR = H / HKV, b = row / H, h = row % H;
  const long part = (long)(b * HKV + h / GR) * NS * GR + h % GR;
  float m = -1e30f, l = 0.f;
  if (lane < NS) {
    m = pml[(part + (long)lane * GR) * 2];
    l = pml[(part + (long)lane * GR) * 2 + 1];
  }
  const float M = wave_reduce_max(m);
  const float a = lane < NS ? __builtin_amdgcn_exp2f(m - M) : 0.f;
  const float sum = wave_reduce_sum(l * a);
  float o[DPL];
#pragma unroll
  for (int i = 0; i < DPL; ++i) o[i] = 0.f;
#pragma unroll 8
  for (int s = 0; s < NS; ++s) {
    const float w = __builtin_bit_cast(
        float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, a), s));
#pragma unroll
    for (int i = 0; i < DPL; ++i)
      o[i] += w * pacc[(part + (long)s * GR) * D + lane * DPL + i];
  }
  const float inv = sum > 0.f ? 1.f / sum : 0.f;
#pragma unroll
  for (int i = 0; i < DPL; ++i)
    out[(long)row * D + lane * DPL + i] = f2bf(o[i] * inv);
}

// step: a decode step's projections in the place of q, NS the shares of all
// sequences; arrived: a zero for every B * HKV * groups of 16 query heads
static void pa_launch(const void* q, long q_stride, const PaStep* step,
                      void* kcache, void* vcache, const int* block_table,
                      const int* ctx_len, void* out, void* pacc, void* pml,
                      int* arrived, int B, int H, int HKV, int D,
                      int max_blocks, int NS, float scale, bool fp8,
                      bool aligned, hipStream_t stream) {
  const int GR = H / HKV, NG = (GR + 15) / 16;
  const PaStep in = step != nullptr ? *step : PaStep{};
  const int grid =
      (step != nullptr ? 1 : B) * HKV * NG * NS + in.ahead.blocks;
#define PA(DD, F8, AL, R, ST)                                                 \
  hipLaunchKernelGGL((paged_attn_kernel<DD, F8, AL, R, ST>), dim3(grid),      \
                     dim3(256), pa_lds(DD, R) + (ST ? 18 * DD * 2 : 0), stream, \
                     (const unsigned short*)q, q_stride, in, (char*)kcache,   \
                     (char*)vcache, block_table, ctx_len,                     \
                     (unsigned short*)out, (float*)pacc, (float*)pml,         \
                     arrived, B, H, HKV, max_blocks, NS, scale)
// Tiles in a wave's ring. Two tiles of 128 columns leave a CU to one workgroup;
// from 1024 workgroups on, four for every CU, a second one on the CU counts for
// more, for short contexts are a chain of three reads each. In us, 64 x 32 heads
// of 128, contexts of 16, of 200, of 200 to 2027: two tiles 30, 51, 211; one 20,
// 40, 213 (two waves 12, 38, 217 to 226: the long ones wait for each other).
// 64 x 8 heads, grouped: two 8.8, 16.9, 53; one 6.4, 14.6, 55. With heads of 64,
// 64 x 32: four tiles 22, 38, 120; two 14, 24, 109. A decode step's workgroups wait
// longer, for their share and their rotated queries, so a second one is worth more:
// us a layer, 8 key heads, two tiles and one, contexts of 16, of 200, of 100 to 500,
// of 200 to 2048: 64 sequences 12.3, 22.0, 26.1, 60.2 and 8.9, 18.4, 24.3, 65.5; 66
// 16.5, 28.2, 30.2, 66.1 and 12.2, 23.3, 24.6, 67.1 (three launches 15.2, 25.7, 27.0,
// 67.8); 80 16.9, 29.1, 34.0, 79.3 and 12.6, 24.9, 30.8, 76.9; 112 21.7, 38.1, 45.0,
// 105 and 15.0, 30.2, 37.9, 102. Of fp8 pages, which always have one, the step is the
// slower one for many short contexts (128 of 200 25.4, three launches 23.0) and the
// faster one for mixed ones (80 of 200 to 2048 43, 52).
#define PA_D(DD, ST)                                                  \
  do {                                                                \
    if (fp8) PA(DD, true, true, 1, ST);                               \
    else if (!aligned) PA(DD, false, false, 1, ST);                   \
    else if (DD == 128 && B * HKV * NG >= (ST ? 513 : 1024))          \
      PA(DD, false, true, 1, ST);                                     \
    else PA(DD, false, true, 2, ST);                                  \
  } while (0)
  if (step != nullptr) {
    if (D == 64) PA_D(64, true);
    else PA_D(128, true);
  } else {
    if (D == 64) PA_D(64, false);
    else PA_D(128, false);
  }
#undef PA_D
#undef PA
}

extern "C" void launch_paged_attn(const void* q, long q_stride, void* kcache,
                                  void* vcache, const int* block_table,
                                  const int* ctx_len, void* out, void* pacc,
                                  void* pml, int B, int H, int HKV, int D,
                                  int max_blocks, int NS, float scale,
                                  bool fp8, bool aligned, hipStream_t stream) {
  pa_launch(q, q_stride, nullptr, kcache, vcache, block_table, ctx_len, out,
            pacc, pml, nullptr, B, H, HKV, D, max_blocks, NS, scale, fp8,
            aligned, stream);
  if (NS > 1) {
    const int rows = B * H;
#define PC(DD)                                                                \
  hipLaunchKernelGGL(paged_attn_combine_kernel<DD>, dim3((rows + 3) / 4),     \
                     dim3(256), 0, stream, (const float*)pacc,                \
                     (const float*)pml, (unsigned short*)out, rows, H, HKV,   \
                     NS)
    if (D == 64) PC(64);
    else PC(128);
#undef PC
  }
}

extern "C" void launch_step_attn(const void* qkv, const float* parts, int S,
                                 const void* bias, const float* cs,
                                 const float* sn, void* kcache, void* vcache,
                                 const int* block_table, const int* ctx_len,
                                 void* out, void* pacc, void* pml,
                                 int* arrived, const int* slots, int G, int B,
                                 int H, int HKV, int D, int max_blocks,
                                 float scale, bool fp8, bool aligned,
                                 const Ahead* ahead, hipStream_t stream) {
  const PaStep step = {(const unsigned short*)qkv, parts, S,
                       (const unsigned short*)bias, cs, sn, slots,
                       *ahead};
  pa_launch(nullptr, 0, &step, kcache, vcache, block_table, ctx_len, out, pacc,
            pml, arrived, B, H, HKV, D, max_blocks, G, scale, fp8, aligned,
            stream);
}

// Who takes what in the attention launches of a decode step, which know the
// lengths only on the device. `wide` and `narrow` are the shares of a head group
// that fill the CUs with one workgroup and, of fp8 pages, with two (else 0).
//  - Up to 7/8 of that many sequences are cut into tiles of 32 keys so that all shares
//    run at once and the largest is as small as can be (256 sizes are tried); of
//    fp8 pages no further than 8 tiles where one workgroup a CU does with less.
//  - Of more sequences only those are cut that are above one and a half times
//    what a CU has to read; a CU alone reads nearly twice as fast as all at once.
//  - The largest come first: a CU that got a long one late is what all the
//    others waited for.
// Measured, us in a graph, 32 heads on 8 of 128, equal shares in the batch's
// order and these (bf16; fp8), lengths spread evenly and mixed: 8 of 200 to 4096
// 20.3 -> 17.1 (14.4 -> 13.9); of 200 to 2048, 20 30.6 -> 21.9 (17.9 -> 15.7), 30
// 32.9 -> 30.7 (23 -> 20.5), 42 46.4 -> 36.2 (38.5 -> 23.6), 64 60.5 -> 51.1 (37.4
// -> 33.7); lengths all alike take what they took. One launch per step, 5 us, which
// clears the counters of all layers too, as one did before.
// A sequence is cut at 4 tiles or more, one for each wave, into 32 shares or less;
// the shares are then made even, so that n of them have more than 4 (n - 1) tiles (5
// tiles are shares of 3 and 2). asked > 0: that many for each.
__host__ __device__ constexpr bool plan_many(int B, int p) {
  return B > p - p / 8;
}
constexpr int PLAN_ROWS = 1024;  // beyond, each sequence is a share, in order

// What else a step begins with, in workgroups of the same launch: the RMS norm of its
// rows x. (A launch of its own costs 3 to 4 us of a step.) Sums as in
// norm_fwd_small_kernel.
struct PlanRows {
  const unsigned short *x, *w;
  unsigned short* h;
  int H;  // a multiple of 8, up to 8192; 0: none
  float eps;
};
__device__ __forceinline__ void plan_row(const PlanRows& p, int row) {
  __shared__ float red[4];
  const int tid = threadIdx.x;
  s16x8 xv[4];
  float sumsq = 0.f;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int c = (tid + k * 256) * 8;
    if (c < p.H) {
      xv[k] = *reinterpret_cast<const s16x8*>(p.x + (long)row * p.H + c);
      float f[8];
      bf8_to_f32(xv[k], f);
#pragma unroll
      for (int i = 0; i < 8; ++i) sumsq += f[i] * f[i];
    }
  }
  sumsq = wave_reduce_sum(sumsq);
  if ((tid & 63) == 0) red[tid >> 6] = sumsq;
  __syncthreads();
  const float inv =
      rsqrtf((red[0] + red[1] + red[2] + red[3]) / p.H + p.eps);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int c = (tid + k * 256) * 8;
    if (c < p.H) {
      float f[8], wf[8];
      bf8_to_f32(xv[k], f);
      bf8_to_f32(*reinterpret_cast<const s16x8*>(p.w + c), wf);
      s16x8 o;
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = (short)f2bf(f[i] * inv * wf[i]);
      *reinterpret_cast<s16x8*>(p.h + (long)row * p.H + c) = o;
    }
  }
}

__global__ void __launch_bounds__(256)
step_plan_kernel(const int* __restrict__ ctx, const int* __restrict__ table,
                 int B, int max_blocks, int G, int narrow, int wide, int asked,
                 int4* __restrict__ slots, int* __restrict__ arrived,
                 long zeros, int clear, const PlanRows rows) {
  const int tid = threadIdx.x;
  if (blockIdx.x > clear + (B + 3) / 4) {
    plan_row(rows, blockIdx.x - 1 - clear - (B + 3) / 4);
    return;
  }
  if (blockIdx.x > clear) {
    // a wave for each row: does another one put a token into a page that it
    // reads, ahead of its own
    const int i = (blockIdx.x - 1 - clear) * 4 + (tid >> 6);
    if (i >= B) return;
    const int pos = ctx[i] - 1;
    bool found = false;
    for (int j = tid & 63; j < B; j += 64) {
      const int p = ctx[j] - 1, pg = p / PBLK;
      if (j != i && p >= 0 && p < pos && pg < max_blocks)
        found |= table[(long)i * max_blocks + pg] ==
                 table[(long)j * max_blocks + pg];
    }
    found = __any(found);
    if ((tid & 63) == 0) reinterpret_cast<int*>(slots)[i * 8 + 6] = found;
    return;
  }
  if (blockIdx.x > 0) {
    for (long i = (blockIdx.x - 1) * 256L + tid; i < zeros; i += clear * 256L)
      arrived[i] = 0;
    return;
  }
  // (of the second four of a share's numbers two are other workgroups')
  auto of_sequence = [&](int slot, int first, int n) {
    *reinterpret_cast<int2*>(slots + slot * 2 + 1) = int2{first, n};
  };
  auto length = [&](int b) { return min(max(ctx[b], 0), max_blocks * PBLK); };
  if (B > PLAN_ROWS) {
    for (int i = tid; i < G; i += 256) {
      const bool is = i < B;
      slots[i * 2] = int4{is ? i : -1, is ? ctx[i] : 0, 0,
                          is ? (length(i) + KT - 1) / KT : 0};
      of_sequence(i, i, 1);
    }
    return;
  }
  int* tiles = reinterpret_cast<int*>(smem);  // [B]
  int* some = tiles + B;                      // [B]: shares
  int* each = some + B;                       // [B]: tiles of a share
  __shared__ int sum, most, best[2];
  if (tid == 0) sum = most = 0, best[0] = best[1] = 1 << 30;
  __syncthreads();
  int s = 0, m = 0;
  for (int b = tid; b < B; b += 256) {
    const int t = (length(b) + KT - 1) / KT;
    tiles[b] = t;
    s += t;
    m = max(m, t);
  }
  // (256 threads' atomics on one number were half of the launch)
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    s += __shfl_xor(s, off, 64);
    m = max(m, __shfl_xor(m, off, 64));
  }
  if ((tid & 63) == 0) {
    atomicAdd(&sum, s);
    atomicMax(&most, m);
  }
  __syncthreads();
  // tiles of a share so that there are p shares or less; of many sequences, two
  // thirds of p more than them. Quotients by a multiplication, exact below 2^16
  // tiles and never too small: the largest size is always one that does.
  auto cut = [&](int p, int* found) {
    if (plan_many(B, p)) return (3 * sum + 2 * p - 1) / (2 * p);
    const int lo = max((sum + p - 1) / p, NW), hi = max(most, lo);
    const int c = lo + (int)(((long)(hi - lo) * tid + 254) / 255);
    const unsigned int inv = 0xffffffffu / (unsigned)c + 1;
    int n = 0;
    for (int b = 0; b < B; ++b)
      n += max((int)__umulhi((unsigned)(tiles[b] + c - 1), inv), 1);
    const unsigned long long does = __ballot(n <= p);
    if (does) {
      const int least = __shfl(c, __ffsll(does) - 1, 64);
      if ((tid & 63) == 0) atomicMin(found, least);
    }
    __syncthreads();
    return min(*found, hi);
  };
  int c = 1;
  if (asked <= 0) {
    c = cut(narrow, &best[0]);
    if (wide > 0) c = max(cut(wide, &best[1]), min(c, 8));
    c = max(max(c, NW), (most + 31) / 32);
  }
  for (int b = tid; b < B; b += 256) {
    const int t = tiles[b], n = asked > 0 ? asked : max((t + c - 1) / c, 1);
    const int per = max((t + n - 1) / n, 1);
    some[b] = asked > 0 ? n : max((t + per - 1) / per, 1);
    each[b] = per;
  }
  __syncthreads();
  int all = 0;
  for (int b = tid; b < B; b += 256) {
    const int t = tiles[b], n = some[b], per = each[b];
    int first = 0;
    all = 0;
    for (int j = 0; j < B; ++j) {
      const int nj = some[j], pj = each[j];
      all += nj;
      if (pj > per || (pj == per && j < b)) first += nj;
    }
    for (int i = 0; i < n && first + i < G; ++i) {
      slots[(first + i) * 2] =
          int4{b, ctx[b], min(i * per, t), min((i + 1) * per, t)};
      of_sequence(first + i, first, n);
    }
  }
  // thread 0 has a sequence
  if (tid == 0) sum = all;
  __syncthreads();
  for (int i = sum + tid; i < G; i += 256) slots[i * 2] = int4{-1, 0, 0, 0};
}

// Shares that a launch has room for; asked is taken up to PLAN_ROWS sequences.
extern "C" int step_plan_room(int B, int narrow, int wide, int asked) {
  if (B > PLAN_ROWS) return B;
  if (asked > 0) return B * asked;
  const int p = std::max(narrow, wide);
  return plan_many(B, p) ? B + 2 * p / 3 : p;
}

extern "C" void launch_step_plan(const int* ctx, const int* table, int B,
                                 int max_blocks, int G, int narrow, int wide,
                                 int asked, int* slots, int* arrived,
                                 long zeros, const void* x, const void* w,
                                 void* h, int H, float eps,
                                 hipStream_t stream) {
  const int clear = (int)std::min((zeros + 1023) / 1024, 256L);
  const PlanRows rows = {(const unsigned short*)x, (const unsigned short*)w,
                         (unsigned short*)h, H, eps};
  hipLaunchKernelGGL(step_plan_kernel,
                     dim3(1 + clear + (B + 3) / 4 + (H > 0 ? B : 0)),
                     dim3(256), B > PLAN_ROWS ? 0 : B * 12, stream, ctx, table,
                     B, max_blocks, G, narrow, wide, asked, (int4*)slots,
                     arrived, zeros, clear, rows);
}

// Write one new token's K/V into the paged cache (decode step).
// knew/vnew: [B, HKV, D] bf16; slot[b] = ctx position of the new token.
template <int D, typename CT>
__global__ void __launch_bounds__(256)
cache_put_kernel(const unsigned short* __restrict__ knew,
                 const unsigned short* __restrict__ vnew,
                 CT* __restrict__ kcache,
                 CT* __restrict__ vcache,
                 const int* __restrict__ block_table,
                 const int* __restrict__ slot, int B, int HKV,
                 int max_blocks) {
  const long total = (long)B * HKV * D;
  const long stride = (long)gridDim.x * blockDim.x;
  const long blk_stride = (long)HKV * PBLK * D;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += stride) {
    const int d = (int)(i % D);
    const int kvh = (int)((i / D) % HKV);
    const int b = (int)(i / ((long)D * HKV));
    const int pos = slot[b];
    const int blk = block_table[(long)b * max_blocks + pos / PBLK];
    const long off =
        (long)blk * blk_stride + ((long)kvh * PBLK + pos % PBLK) * D + d;
    cache_store(kcache + off, knew[i]);
    cache_store(vcache + off, vnew[i]);
  }
}

extern "C" void launch_cache_put(const void* knew, const void* vnew,
                                 void* kcache, void* vcache,
                                 const int* block_table, const int* slot,
                                 int B, int HKV, int D, int max_blocks,
                                 bool fp8, hipStream_t stream) {
  const long total = (long)B * HKV * D;
  int blocks = (int)min((total + 255) / 256, (long)2048);
#define CP(DD, CT)                                                             \
  hipLaunchKernelGGL((cache_put_kernel<DD, CT>), dim3(blocks), dim3(256), 0,   \
                     stream, (const unsigned short*)knew,                      \
                     (const unsigned short*)vnew, (CT*)kcache, (CT*)vcache,    \
                     block_table, slot, B, HKV, max_blocks)
  if (D == 64) {
    if (fp8) CP(64, unsigned char); else CP(64, unsigned short);
  } else {
    if (fp8) CP(128, unsigned char); else CP(128, unsigned short);
  }
#undef CP
}

// A decode step's projections qkv [B, H + 2 HKV, D] on their way, for callers
// that attend by themselves (the attention kernel does this too): queries and
// keys are rotated by the position ctx - 1 of the new token (half-split, fp32,
// tables [positions, D / 2]); queries go to q [B, H, D], keys and values to
// their place in the cache. One launch for what a rotation, three copies and
// a cache write took (5 launches of 4 us each, in a graph). A thread has
// columns c .. c + 3 of either half of a head. With S > 0 the projections come
// as the S fp32 slabs of a product whose K was shared, and are summed, given
// their bias and rounded here: a launch less (product of 6144 x 4096 and this,
// in a graph, 64 rows 20.8 -> 18.6 us, 17 rows 18.4 -> 15.7).
template <int D, typename CT>
__global__ void __launch_bounds__(256)
rope_put_kernel(const PaStep p, const int* __restrict__ ctx,
                unsigned short* __restrict__ q,
                CT* __restrict__ kcache, CT* __restrict__ vcache,
                const int* __restrict__ block_table, int B, int H, int HKV,
                int max_blocks) {
  constexpr int PER = D / 8;  // threads of a head
  const int heads = H + 2 * HKV;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)B * heads * PER) return;
  const int c = (int)(i % PER) * 4;
  const int h = (int)(i / PER % heads), b = (int)(i / PER / heads);
  const int pos = ctx[b] - 1;
  unsigned short a[4], e[4];
  step_columns<D>(p, B, heads, b, h, c, h < H + HKV, pos, a, e);
  if (h < H) {
    unsigned short* o = q + ((long)b * H + h) * D + c;
    *reinterpret_cast<i32x2*>(o) = *reinterpret_cast<const i32x2*>(a);
    *reinterpret_cast<i32x2*>(o + D / 2) = *reinterpret_cast<const i32x2*>(e);
    return;
  }
  const int kvh = (h - H) % HKV;
  CT* o = (h < H + HKV ? kcache : vcache) +
          (((long)block_table[(long)b * max_blocks + pos / PBLK] * HKV + kvh) *
               PBLK + pos % PBLK) * D + c;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    cache_store(o + j, a[j]);
    cache_store(o + D / 2 + j, e[j]);
  }
}

extern "C" void launch_rope_put(const void* qkv, const float* parts, int S,
                                const void* bias, const float* cs,
                                const float* sn, const int* ctx, void* q,
                                void* kcache, void* vcache,
                                const int* block_table, int B, int H, int HKV,
                                int D, int max_blocks, bool fp8,
                                hipStream_t stream) {
  const long total = (long)B * (H + 2 * HKV) * (D / 8);
  const PaStep p = {(const unsigned short*)qkv, parts, S,
                    (const unsigned short*)bias, cs, sn};
#define RP(DD, CT)                                                            \
  hipLaunchKernelGGL((rope_put_kernel<DD, CT>), dim3((total + 255) / 256),    \
                     dim3(256), 0, stream, p, ctx, (unsigned short*)q,        \
                     (CT*)kcache, (CT*)vcache,            \
                     block_table, B, H, HKV, max_blocks)
  if (D == 64) {
    if (fp8) RP(64, unsigned char); else RP(64, unsigned short);
  } else {
    if (fp8) RP(128, unsigned char); else RP(128, unsigned short);
  }
#undef RP
}
