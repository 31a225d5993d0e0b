// MFMA attention of single-token rows over paged bf16 latents (see
// latent_attention.hip for the mechanism, the cache layout and the row
// arguments; that file's one-head kernel covers the other types and ranks).
//
// A workgroup serves HG groups of 16 heads of one row, so a latent is read
// from HBM once for all of them; the visible keys of a row are split over NS
// workgroups whose partial results a second kernel joins.
//
// Cache rows and queries have RR = R + ROT numbers, of which all take part in
// the scores and the first R are the value. The same bytes are key and value,
// so a tile of 64 keys goes to LDS once, as it lies in the cache, by
// global_load_lds (the next tile's loads are in flight behind the current
// one); values are transposed on their way out of LDS.
//  - scores: each of the 4 waves of a head group has 16 keys (one page) and
//    a softmax state of its own;
//  - the waves exchange their weights and maxima through LDS;
//  - output: each wave has R / 4 latent columns, for all keys. A weight goes in
//    as the sum of two bf16 numbers: with one, a tile of 64 keys, which has
//    fewer weights of exactly 1 than two of 32 had, was 0.3 to 1.3% further off
//    64 bits than those (2.0e-3 of the result; with two 1.66e-3, what its own
//    rounding leaves). Up to 11% of the kernel at many keys.
// Both products are mfma_f32_16x16x32_bf16 with keys (then latent columns) as
// rows and heads as columns, so that states and rescaling are lane-local; a
// lane's weights of the exchange are its operand of the second product.
//
// At many keys bound by reading the cache, at few by the chain through a tile
// (0.7 us of it barriers, maxima and exchange) and the join. One wave
// for two head groups reads LDS half as often, but has nobody to fill its
// waits: 2.9 us a tile against 1.9. Tiles of 32 keys that passed through
// registers and were kept twice, one copy transposed, with 64 heads in a
// workgroup, took (rank 512, 32 heads, us, then and now) 1 row of 2048 keys
// 28 -> 17, 32 rows of 300 to 2048 37 -> 25.5, 16 of 100 to 4000 46 -> 25.5, 64
// of 200 to 2000 43 -> 36; 64 heads: 32 rows of 2048 40 -> 35, 64 rows of 200 to
// 2000 51 -> 51, for the second group of 32 heads reads the tiles from L2.
#include "common.h"

#define PBLK 16
#define KT 64  // keys of a tile: a page for each wave
#define LOG2E 1.4426950408889634f

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

extern __shared__ __attribute__((aligned(16))) char smem[];

union ld_frag {
  bf16x8 v;
  s16x4 h[2];
  unsigned int d[4];
};

__device__ __forceinline__ unsigned int ld_pack(float a, float b) {
  return __builtin_bit_cast(
      unsigned int, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

// LDS of the workgroup is done with what it read or written by all
__device__ __forceinline__ void ld_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Where the 16-byte piece c of row r of R numbers lies in the row. Pieces are
// read by 16 rows at a time (keys) and by 4 rows x 2 neighbours (values): the
// low bits of the row move pairs, the next one swaps within a pair.
template <int R>
__device__ __forceinline__ int ld_piece(int r, int c) {
  return R % 128 == 0 ? c ^ ((r & 7) << 1 | (r >> 3 & 1))
                      : c ^ ((r & 3) << 1 | (r >> 2 & 1));
}

// Weight of a row's sum: 1 / l with the softmax's state m (log2 units), l and
// the sink of the head, times its gate.
__device__ __forceinline__ float row_weight(float m, float l, long row,
                                            int head, const float* sink,
                                            const unsigned short* gate,
                                            int ld_gate) {
  float inv = l > 0.f ? 1.f / l : 0.f;
  if (sink != nullptr && l > 0.f) {
    const float s = sink[head] * LOG2E, top = fmaxf(m, s);
    const float a = __builtin_amdgcn_exp2f(m - top);
    inv = a / (l * a + __builtin_amdgcn_exp2f(s - top));
  }
  if (gate != nullptr) inv *= sigmoid_exact(bf2f(gate[row * ld_gate + head]));
  return inv;
}

template <int R, int ROT, int HG>
constexpr int ld_lds() {
  return 2 * KT * (R + ROT) * 2 + 4 * HG * (1024 + 64);
}

// ALIGNED: the cache starts at a multiple of 16 bytes, as the copies to LDS ask;
// else its rows pass through registers, one tile after another.
template <int R, int ROT, int HG, bool ALIGNED = true>
__global__ void __launch_bounds__(256 * HG, R + ROT <= 256 ? 2 * HG : HG)
latent_decode_kernel(const unsigned short* __restrict__ q,
                     const unsigned short* __restrict__ cache,
                     const int* __restrict__ block_table,
                     const int* __restrict__ row_seq,
                     const int* __restrict__ ctx,
                     unsigned short* __restrict__ out,
                     float* __restrict__ pacc, float* __restrict__ pml,
                     int M, int H, int NG, int NS, int max_blocks, int window,
                     float scale, const float* __restrict__ sink,
                     const unsigned short* __restrict__ gate, int ld_gate) {
  static_assert(ROT == 0 || ROT == 64, "eight 16-byte pieces per key");
  constexpr int RR = R + ROT;
  constexpr int MAIN = KT * R * 2;  // of a buffer; its key parts follow
  constexpr int BUF = KT * RR * 2;
  constexpr int RP = R / 8;         // 16-byte pieces of a row
  constexpr int NP = R / 32 / HG;   // copies of a wave: 16 / HG rows' values
  constexpr int NR = ROT / 32 / HG; // and their key parts
  constexpr int QS = R / 32, TS = ROT / 32;  // score steps
  constexpr int OB = R / 64;        // output blocks of a wave

  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int w = wid & 3, hg = wid >> 2;  // page of the tile, head group
  const int c16 = lane & 15, g = lane >> 4;
  // the workgroups of the same keys follow on one XCD, which reads them once
  const int share = blockIdx.x / (8 * NG) * 8 + blockIdx.x % 8;
  const int grp = blockIdx.x / 8 % NG;
  const int split = share % NS, row = share / NS;
  if (row >= M) return;
  const int head0 = grp * HG * 16;
  float* weights =
      reinterpret_cast<float*>(smem + 2 * BUF) + hg * 4 * 256;
  float* maxima =
      reinterpret_cast<float*>(smem + 2 * BUF) + HG * 4 * 256 + hg * 64;

  // queries pass through the second buffer
  char* qb = smem + BUF;
  auto from = [&](int r) {
    return q + ((long)row * H + min(head0 + r, H - 1)) * RR;
  };
  for (int p = wid; p < HG * QS; p += 4 * HG) {
    const int at = p * 64 + lane, r = at / RP, c = at % RP;
    copy_to_lds(from(r) + ld_piece<R>(r & 15, c) * 8, qb + p * 1024);
  }
  for (int p = wid; p < HG * TS; p += 4 * HG) {
    const int r = p * 8 + (lane >> 3), c = (lane & 7) ^ (r & 7);
    copy_to_lds(from(r) + R + c * 8, qb + MAIN + p * 1024);
  }

  const int L = min(ctx[row], max_blocks * PBLK);
  const int lo = L > window ? L - window : 0;
  const int T0 = lo / KT, T1 = L > 0 ? (L + KT - 1) / KT : T0;
  const int per = (T1 - T0 + NS - 1) / NS;
  const int ts = T0 + split * per, te = min(T1, ts + per);
  const int last_page = L > 0 ? (L - 1) / PBLK : 0;
  const int* bt = block_table + (long)row_seq[row] * max_blocks;

  // page w of each of the next 64 tiles, on the lanes; the window's first page
  // in the place of those ahead of it, which may be in use elsewhere
  int pages = 0;
  auto fetch_pages = [&](int t) {
    pages = bt[max(min((t + lane) * 4 + w, last_page), lo / PBLK)];
  };
  auto issue = [&](int t) {
    if (((t - ts) & 63) == 0) fetch_pages(t);
    const unsigned short* src =
        cache +
        (long)__builtin_amdgcn_readlane(pages, (t - ts) & 63) * PBLK * RR;
    char* dst = smem + ((t - ts) & 1) * BUF;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int p = hg * NP + i;
      const int at = p * 64 + lane, r = at / RP, c = at % RP;
      to_lds<ALIGNED>(src + r * RR + ld_piece<R>(r, c) * 8,
                      dst + (w * NP * HG + p) * 1024);
    }
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int p = hg * NR + i;
      const int r = p * 8 + (lane >> 3), c = (lane & 7) ^ (r & 7);
      to_lds<ALIGNED>(src + r * RR + R + c * 8,
                      dst + MAIN + (w * NR * HG + p) * 1024);
    }
  };

  constexpr int COPIES = ALIGNED ? NP + NR : 0;  // in flight, of a tile
  bf16x8 qf[QS + TS];
  if (ts < te) {
    issue(ts);
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(COPIES) : "memory");
    ld_barrier();
#pragma unroll
    for (int s = 0; s < QS; ++s)
      qf[s] = *reinterpret_cast<const bf16x8*>(
          qb + (hg * 16 + c16) * (R * 2) +
          ld_piece<R>(c16, s * 4 + g) * 16);
#pragma unroll
    for (int s = 0; s < TS; ++s)
      qf[QS + s] = *reinterpret_cast<const bf16x8*>(
          qb + MAIN + (hg * 16 + c16) * (ROT * 2) +
          (((s * 4 + g) ^ (c16 & 7)) * 16));
    ld_barrier();
    if (ts + 1 < te) {
      issue(ts + 1);
      asm volatile("s_waitcnt vmcnt(%0)" ::"i"(COPIES) : "memory");
    }
  }
  if (ts + 1 >= te) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  const float scale2 = scale * LOG2E;
  float m = -1e30f, l = 0.f;  // of the sums, l: of this lane's keys
  float mw = -1e30f;          // the largest of this wave's keys
  f32x4 acc[OB];
#pragma unroll
  for (int i = 0; i < OB; ++i) acc[i] = {0.f, 0.f, 0.f, 0.f};

  for (int t = ts; t < te; ++t) {
    char* buf = smem + ((t - ts) & 1) * BUF;
    const int key0 = t * KT + w * 16;
    if (key0 + 16 > L || key0 + 16 <= lo) {
      // what lies behind the last key, or was copied in the place of a page
      // ahead of the window, must not meet its zero weight; each wave clears
      // what it copied
      const int from = key0 + 16 <= lo ? 0 : max(L - key0, 0);
      for (int at = max(from * (R * 2), hg * NP * 1024) + lane * 16;
           at < (hg + 1) * NP * 1024; at += 1024)
        *reinterpret_cast<i32x4*>(buf + w * (QS * 1024) + at) =
            i32x4{0, 0, 0, 0};
    }
    // this tile is there and the other buffer is free
    ld_barrier();
    if (t > ts && t + 1 < te) issue(t + 1);

    // scores of my 16 keys, in two chains
    f32x4 sc = {0.f, 0.f, 0.f, 0.f}, sc2 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < QS + TS; ++s) {
      const char* a =
          s < QS ? buf + (w * 16 + c16) * (R * 2) +
                       ld_piece<R>(c16, s * 4 + g) * 16
                 : buf + MAIN + (w * 16 + c16) * (ROT * 2) +
                       ((((s - QS) * 4 + g) ^ (c16 & 7)) * 16);
      const bf16x8 kf = *reinterpret_cast<const bf16x8*>(a);
      f32x4& to = s & 1 ? sc2 : sc;
      to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[s], to, 0, 0, 0);
    }
    float top = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int key = key0 + g * 4 + r;
      sc[r] = key >= lo && key < L ? (sc[r] + sc2[r]) * scale2 : -INFINITY;
      top = fmaxf(top, sc[r]);
    }
    top = lanes_max<32>(lanes_max<16>(top));
    mw = fmaxf(mw, top);
#pragma unroll
    for (int r = 0; r < 4; ++r) sc[r] = __builtin_amdgcn_exp2f(sc[r] - mw);
    *reinterpret_cast<f32x4*>(weights + (w * 64 + lane) * 4) = sc;
    if (g == 0) maxima[w * 16 + c16] = mw;
    ld_barrier();

    // all weights, relative to the largest maximum so far
    ld_frag pf[2], pl[2];  // high and low parts
    float mx[4], ma = m;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      mx[i] = maxima[i * 16 + c16];
      ma = fmaxf(ma, mx[i]);
    }
    if (!__all(ma <= m)) {
      const float alpha = __builtin_amdgcn_exp2f(m - ma);
      m = ma;
      l *= alpha;
#pragma unroll
      for (int i = 0; i < OB; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][r] *= alpha;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x4 p =
          *reinterpret_cast<const f32x4*>(weights + (i * 64 + lane) * 4);
      const float f = __builtin_amdgcn_exp2f(mx[i] - m);
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float a = p[e * 2] * f, b = p[e * 2 + 1] * f;
        l += a + b;
        const unsigned int h = ld_pack(a, b);
        pf[i >> 1].d[(i & 1) * 2 + e] = h;
        pl[i >> 1].d[(i & 1) * 2 + e] =
            ld_pack(a - __builtin_bit_cast(float, h << 16),
                    b - __builtin_bit_cast(float, h & 0xffff0000u));
      }
    }
    // keys 4 g .. 4 g + 3 of two pages at a time, as the weights lie
    const int vr = g * 4 + (c16 >> 2);
#pragma unroll
    for (int i = 0; i < OB; ++i) {
      const int c = (w * OB + i) * 2 + (c16 >> 1 & 1);
      const char* a =
          buf + vr * (R * 2) + ld_piece<R>(vr, c) * 16 + (c16 & 1) * 8;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        ld_frag vf;
#pragma unroll
        for (int e = 0; e < 2; ++e)
          vf.h[e] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) s16x4*)(
                  a + (kb * 2 + e) * (16 * R * 2)));
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.v, pf[kb].v,
                                                         acc[i], 0, 0, 0);
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.v, pl[kb].v,
                                                         acc[i], 0, 0, 0);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }

  // (every wave has the weights of all keys)
  l = lanes_sum<32>(lanes_sum<16>(l));
  const int head = head0 + hg * 16 + c16;
  if (head >= H) return;
  const long rh = (long)row * H + head;
  const int col = w * (OB * 16) + g * 4;
  if (NS == 1) {
    const float inv = row_weight(m, l, row, head, sink, gate, ld_gate);
#pragma unroll
    for (int i = 0; i < OB; ++i) {
      const i32x2 o = {(int)ld_pack(acc[i][0] * inv, acc[i][1] * inv),
                       (int)ld_pack(acc[i][2] * inv, acc[i][3] * inv)};
      *reinterpret_cast<i32x2*>(out + rh * R + col + i * 16) = o;
    }
  } else {
    const long part = rh * NS + split;
#pragma unroll
    for (int i = 0; i < OB; ++i)
      *reinterpret_cast<f32x4*>(pacc + part * R + col + i * 16) = acc[i];
    if (g == 0 && w == 0) {
      pml[part * 2] = m;
      pml[part * 2 + 1] = l;
    }
  }
}

// Join NS <= 64 partial results: a wave per (row, head) and 256 columns, the
// shares' states on its lanes. With a wave per (row, head) that went through
// the states one by one: 32 rows of 32 heads, 8 shares of rank 512, 12.7 us,
// now 4.8.
__global__ void __launch_bounds__(256)
latent_combine_kernel(const float* __restrict__ pacc,
                      const float* __restrict__ pml,
                      unsigned short* __restrict__ out, int RH, int R,
                      int NS, int H, const float* __restrict__ sink,
                      const unsigned short* __restrict__ gate, int ld_gate) {
  const int lane = threadIdx.x & 63;
  const int parts = (R + 255) / 256;
  const int at = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int rh = at / parts, c = at % parts * 256 + lane * 4;
  if (rh >= RH) return;
  float m = -1e30f, l = 0.f;
  if (lane < NS) {
    m = pml[((long)rh * NS + lane) * 2];
    l = pml[((long)rh * NS + lane) * 2 + 1];
  }
  const float M = wave_reduce_max(m);
  float a = __builtin_amdgcn_exp2f(m - M);
  const float sum = wave_reduce_sum(l * a);
  a *= row_weight(M, sum, rh / H, rh % H, sink, gate, ld_gate);
  const float* p = pacc + (long)rh * NS * R + min(c, R - 4);
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int s = 0; s < NS; ++s) {
    const float w = __builtin_bit_cast(
        float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, a), s));
    const f32x4 v = *reinterpret_cast<const f32x4*>(p + (long)s * R);
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] += w * v[i];
  }
  if (c < R) {
    const i32x2 two = {(int)ld_pack(o[0], o[1]), (int)ld_pack(o[2], o[3])};
    *reinterpret_cast<i32x2*>(out + (long)rh * R + c) = two;
  }
}

// The same join, and the product of the joined latents with the heads' value
// weights W [H, N, R], which is what follows: out[m, h, :] = W[h] latent[m, h]. A
// workgroup has ROWS rows of a head, joined while the weights come to LDS by whole
// lines, and then 16 columns a wave; roundings and sums are those of
// latent_combine_kernel and head_gemm_kernel, bit for bit. Bound by the way of the
// shares and the weights into a CU, of 8 rows 128 KiB each at 8 shares of rank 512 and
// 128 columns: the first shares are on their way ahead of the weights (behind them 10.7
// us for 8.2), and there are 4 rows, two waves each, where those of all still fit the
// card at once. us over fresh weights, 8 and 4 rows, rank 512, 128 columns, 8 shares,
// 32 heads: 1 row 5.9 and 5.0, 32 6.0 and 5.4, with 16 shares 11.2 and 8.5; in two
// rounds, 40 6.1 and 9.1; 128 heads, 8 rows 6.9 and 6.9, 12 8.0 and 11.6; rank 384, 64
// columns, 32 heads, 32 rows 4.5 and 3.9, 40 4.6 and 4.9. us with the attention,
// launches of their own and this of 8 rows, 32 heads: rank 512, 128 columns, 32 rows of
// 2000 keys 33.0, 28.8, one 20.8, 19.3, 64 of 300 23.8, 20.1; rank 256, 64 columns, 32
// of 2000 22.4, 17.5.
// LDS rows' 16-byte pieces are XOR-ed with the row.
constexpr int LV_WAVES = 8;
constexpr int lv_lds(int R, int N, int ROWS) { return (N + ROWS) * R * 2; }

template <int R, int ROWS>
__global__ void __launch_bounds__(LV_WAVES * 64)
latent_values_kernel(const float* __restrict__ pacc,
                     const float* __restrict__ pml,
                     const unsigned short* __restrict__ W,
                     unsigned short* __restrict__ out, int M, int H, int N,
                     int NS, long orow_s, int ohead_s,
                     const float* __restrict__ sink,
                     const unsigned short* __restrict__ gate, int ld_gate) {
  constexpr int RP = R / 8;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int head = blockIdx.x % H, m0 = blockIdx.x / H * ROWS;
  char* xs = smem + N * (R * 2);
  // of 8 rows a wave joins one, of 4 half of one
  constexpr int PARTS = (R + 255) / 256 * ROWS / LV_WAVES, AHEAD = 8;
  static_assert(PARTS * LV_WAVES == (R + 255) / 256 * ROWS, "whole parts");
  const int mine = ROWS == LV_WAVES ? wid : wid % ROWS;
  const int c0 = (ROWS == LV_WAVES ? 0 : wid / ROWS * 256) + lane * 4;
  const long rh = (long)min(m0 + mine, M - 1) * H + head;
  const float* state = pml + (rh * NS + min(lane, NS - 1)) * 2;
  float m = state[0], l = state[1];
  // the first shares are on their way ahead of the weights: loads arrive in order
  f32x4 v[PARTS][AHEAD];
#pragma unroll
  for (int part = 0; part < PARTS; ++part)
#pragma unroll
    for (int s = 0; s < AHEAD; ++s)
      v[part][s] = *reinterpret_cast<const f32x4*>(
          pacc + (rh * NS + min(s, NS - 1)) * R +
          min(part * 256 + c0, R - 4));
  __builtin_amdgcn_sched_barrier(0);
  const unsigned short* from = W + (long)head * N * R;
  for (int p = wid; p < N * RP / 64; p += LV_WAVES) {
    const int at = p * 64 + lane, r = at / RP, c = at % RP;
    copy_to_lds(from + r * R + (c ^ (r & 7)) * 8, smem + p * 1024);
  }
  __builtin_amdgcn_sched_barrier(0);
  if (lane >= NS) m = -1e30f, l = 0.f;
  const float top = wave_reduce_max(m);
  float a = __builtin_amdgcn_exp2f(m - top);
  const float sum = wave_reduce_sum(l * a);
  a *= row_weight(top, sum, rh / H, head, sink, gate, ld_gate);
  auto weight = [&](int s) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, a), s));
  };
#pragma unroll
  for (int part = 0; part < PARTS; ++part) {
    const int c = part * 256 + c0;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < AHEAD; ++s)
      if (s < NS) {
        const float w = weight(s);
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] += w * v[part][s][i];
      }
    const float* p = pacc + rh * NS * R + min(c, R - 4);
#pragma unroll 8
    for (int s = AHEAD; s < NS; ++s) {
      const float w = weight(s);
      const f32x4 x = *reinterpret_cast<const f32x4*>(p + (long)s * R);
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] += w * x[i];
    }
    if (c < R)
      *reinterpret_cast<i32x2*>(xs + mine * (R * 2) +
                                ((c >> 3) ^ mine) * 16 + (c & 4) * 2) =
          i32x2{(int)ld_pack(o[0], o[1]), (int)ld_pack(o[2], o[3])};
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  const int c16 = lane & 15, g = lane >> 4, xrow = c16 & (ROWS - 1);
  for (int n0 = wid * 16; n0 < N; n0 += LV_WAVES * 16) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < R / 32; ++s) {
      const int c = s * 4 + g;
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          *reinterpret_cast<const bf16x8*>(smem + (n0 + c16) * (R * 2) +
                                           (c ^ (c16 & 7)) * 16),
          *reinterpret_cast<const bf16x8*>(xs + xrow * (R * 2) +
                                           (c ^ xrow) * 16),
          acc, 0, 0, 0);
    }
    const int row = m0 + c16;
    if (c16 < ROWS && row < M)
      *reinterpret_cast<i32x2*>(out + row * orow_s + (long)head * ohead_s +
                                n0 + g * 4) =
          i32x2{(int)ld_pack(acc[0], acc[1]), (int)ld_pack(acc[2], acc[3])};
  }
}

// Whether the weights of a head have room in LDS.
extern "C" bool latent_values_fit(int R, int N) {
  return N % 64 == 0 && lv_lds(R, N, 8) <= 160 * 1024;
}

extern "C" void launch_latent_values(const void* pacc, const void* pml,
                                     const void* W, void* out, int M, int H,
                                     int R, int N, int NS, long orow_s,
                                     int ohead_s, const float* sink,
                                     const void* gate, int ld_gate,
                                     hipStream_t stream) {
  // (up to rank 256 a row is one wave's)
  const bool four = R > 256 && (long)H * ((M + 3) / 4) <= 256;
#define LV(RR, ROWS)                                                          \
  hipLaunchKernelGGL((latent_values_kernel<RR, ROWS>),                        \
                     dim3(H * ((M + ROWS - 1) / ROWS)), dim3(LV_WAVES * 64),  \
                     lv_lds(RR, N, ROWS), stream, (const float*)pacc,         \
                     (const float*)pml, (const unsigned short*)W,             \
                     (unsigned short*)out, M, H, N, NS, orow_s, ohead_s,      \
                     sink, (const unsigned short*)gate, ld_gate)
  switch (R) {
    case 64: LV(64, 8); break;
    case 128: LV(128, 8); break;
    case 192: LV(192, 8); break;
    case 256: LV(256, 8); break;
    case 384: if (four) LV(384, 4); else LV(384, 8); break;
    case 512: if (four) LV(512, 4); else LV(512, 8); break;
  }
#undef LV
}

// heads that one workgroup serves
extern "C" int latent_decode_heads(int H) {
  return H <= 16 ? 16 : 32;
}

extern "C" bool latent_decode_covers(int R, int rot) {
  if (rot != 0 && rot != 64) return false;
  return R == 64 || R == 128 || R == 192 || R == 256 || R == 384 || R == 512;
}

extern "C" void launch_latent_decode(
    const void* q, const void* cache, const int* block_table,
    const int* row_seq, const int* ctx, void* out, void* pacc, void* pml,
    int M, int H, int R, int rot, int NS, int max_blocks, int window,
    float scale, const float* sink, const void* gate, int ld_gate,
    bool aligned, bool join, hipStream_t stream) {
  const int heads = aligned ? latent_decode_heads(H) : 16;
  const int ng = (H + heads - 1) / heads;
#define LD(RR, RO, HG, AL)                                                    \
  hipLaunchKernelGGL((latent_decode_kernel<RR, RO, HG, AL>),                  \
                     dim3((M * NS + 7) / 8 * 8 * ng), dim3(256 * HG),         \
                     (ld_lds<RR, RO, HG>()), stream,                          \
                     (const unsigned short*)q, (const unsigned short*)cache,  \
                     block_table, row_seq, ctx, (unsigned short*)out,         \
                     (float*)pacc, (float*)pml, M, H, ng, NS, max_blocks,     \
                     window, scale, sink, (const unsigned short*)gate,        \
                     ld_gate)
#define LD_H(RR, RO)                             \
  do {                                           \
    if (!aligned) LD(RR, RO, 1, false);          \
    else if (heads == 16) LD(RR, RO, 1, true);   \
    else LD(RR, RO, 2, true);                    \
  } while (0)
#define LD_R(RR)              \
  do {                        \
    if (rot == 0) LD_H(RR, 0); \
    else LD_H(RR, 64);        \
  } while (0)
  switch (R) {
    case 64: LD_R(64); break;
    case 128: LD_R(128); break;
    case 192: LD_R(192); break;
    case 256: LD_R(256); break;
    case 384: LD_R(384); break;
    default: LD_R(512); break;
  }
#undef LD_R
#undef LD_H
#undef LD
  if (NS > 1 && join)
    hipLaunchKernelGGL(latent_combine_kernel,
                       dim3((M * H * ((R + 255) / 256) + 3) / 4), dim3(256),
                       0, stream, (const float*)pacc,
                       (const float*)pml, (unsigned short*)out, M * H, R, NS,
                       H, sink, (const unsigned short*)gate, ld_gate);
}
