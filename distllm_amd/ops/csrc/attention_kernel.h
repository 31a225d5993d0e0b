// Fused flash-attention forward for CDNA4 (gfx950), bf16 I/O, fp32 accum.
//
// One kernel family covers the reference's four encoder geometries:
// bidirectional + additive key-pad mask
// (BERT/PubMedBERT, ESM2/ESMC), causal (+GQA) for Mistral/Llama prefill.
// The reference delegated all of this to HF transformers / faesm /
// flash-attn (reference: distllm/embed/encoders/*.py).
//
//  - workgroup = 256 threads = 4 waves; each wave owns 32 q rows
//    (128 q rows per workgroup); KV tiles of 64 keys, double-buffered,
//    ONE barrier per tile.
//  - swapped QK^T: accP = mfma_f32_32x32x16_bf16(A=K, B=Q^T) so each
//    lane holds 32 of the 64 scores of ONE q row -> online softmax is
//    lane-local + one swap of lane halves for the max and one for the sum.
//  - PV is swapped too: accO^T = mfma(A=V^T, B=P): the O accumulator
//    keeps q on lanes, so the alpha rescale is lane-local. The order of
//    the 16 keys of a product is free, so P goes in as the score product
//    left it on the lanes: keys 4h..4h+3 and 8+4h..8+4h+3 of lane half h.
//  - K and V tiles stream by global_load_lds, row by row, their 16-byte
//    (V: 32-byte) pieces XOR-swizzled by the row on the SOURCE address; V is
//    transposed on its way out of LDS (ds_read_b64_tr_b16, 4 keys x 16
//    columns per 16 lanes). Where all rows of a tile exist, they are copied
//    from pointers that the wave shares, at offsets of the lanes that stay.
//  - a tile in which no key is masked for any row of the wave takes the
//    scores as they are: max over the raw products, then one fused multiply
//    and add per exponential.
//  - O leaves by 16-byte stores straight from the accumulators (one lane
//    swap per 8 columns), so that LDS holds the tiles only.
//
// Bound by the vector units (per tile and wave at D = 64: 512 cycles of
// MFMA, about 930 of exponentials, max, sum and conversion, of 1310 in all),
// at a clock of 1.8 GHz that the power allows (the same launch on zeros takes
// 0.77 of the time), and, at D = 128, by LDS reads (32 KB per wave and tile).
// Measured, before (V transposed through registers at D = 64, read element by
// element from memory at 128, every score scaled and masked by itself), then
// (an address of 64-bit products for every copy and lane, 29 more vector
// instructions of 198 per tile) and now: 512 x 512 tokens, 12 heads of 64,
// masked 1240, 594, 565 us (730 TFLOP/s); packed proteins of 64 to 1024, 20
// heads of 64, 248, 196, 187 us with the launch from the host; causal, 32 heads
// of 128 on 8, 16 x 1024 a quarter to all of it 536, 244, 229 us, 4 x 4096
// 2354, 633, 613 (897 TFLOP/s), 2 x 8192 1164, 1107. Four waves a SIMD at
// D = 64 unless the causal compares need more registers (3), two at 128.
// Wave priorities around the products and reading all K or V fragments
// ahead of them measured 0 to 5% slower than leaving the order to the
// compiler.
//
// Layouts: Q [B, SQ, H, D] (token stride parametric), K/V
// [B, SKV, HKV, D] (shared strides), O contiguous BSHD; mask f32
// [B, SKV] additive (0 / -inf) or nullptr. K, V and their strides are
// multiples of 16 bytes.
#pragma once
#include "common.h"
#include <cstdlib>
#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

#define KVBLK 64
#define QWAVE 32
#define LOG2E 1.4426950408889634f

extern __shared__ __attribute__((aligned(16))) char smem[];

union frag_u {
  bf16x8 v;
  s16x4 h[2];
  unsigned int d[4];
};

__device__ __forceinline__ unsigned int pack_bf16(float a, float b) {
  const bf16x2 v = __builtin_convertvector(f32x2{a, b}, bf16x2);
  return __builtin_bit_cast(unsigned int, v);
}

// LDS of a workgroup: two buffers of keys (and their shared part), values
// and mask numbers.
constexpr int attn_lds(int D, int DV, int ROT, bool mask) {
  return 2 * KVBLK * ((D + DV + ROT) * 2 + (mask ? 4 : 0));
}

// VARLEN: Q/K/V are PACKED [total_tokens, H(KV), D] (cu_seqlens int32
// [B+1]); one workgroup per (sequence, q-block, head) via the
// host-built blk_seq/blk_qb map — the protein/fasta path with zero
// padded FLOPs (reference: the faesm flash-attn varlen role,
// distllm/embed/encoders/esm2.py:41-55). Without WINDOW, workgroups past
// nblk * H (nblk = SQa here) zero the rows from cu[Bsz] to SKVa, which no
// sequence holds.
//
// WINDOW (with VARLEN and CAUSAL): the packed queries of a sequence are the
// last ones of its packed keys (cu for queries, cu_k for keys), as when a
// prompt is continued from a cache, and a query sees only the `window`
// latest keys up to its own position. Keys and values may have different
// head sizes (DV) and interleave in one row (tstr_k counts both).
// With ROT, queries have ROT more numbers per head, against ROT numbers of
// each key that all heads share (Kr [Tk, ROT]). sink (a number per head, part
// of the softmax's denominator) and gate (sigmoid of a number per query and
// head on the output) may be null.
//
// With cs and sn (rotation tables [positions, D / 2]; not with WINDOW) queries come
// as they were projected, and are rotated by the angles of pos (a number per query
// row, in Q's order) as they are read, as rope_inplace_kernel would: both halves of
// a head are on the same lane. That saves their way to memory and back, us of
// rotation and attention: packed proteins of 64 to 1024, 20 heads of 64, 124 -> 112
// (114 with the angles asked for ahead of the first tile's copies); causal, 32 heads
// of 128 on 8, 16 x 1024 a quarter to all of it 265 -> 253, 2 x 4096 346 -> 336.
template <int D, bool CAUSAL, bool HAS_MASK, bool VARLEN = false, int DV = D,
          bool WINDOW = false, int ROT = 0>
__global__ void __launch_bounds__(256, D + DV <= 128   ? (CAUSAL ? 3 : 4)
                                       : D + DV <= 256 ? 2
                                                       : 1)
attn_fwd_kernel(const unsigned short* __restrict__ Q,
                const unsigned short* __restrict__ Kt,
                const unsigned short* __restrict__ Vt,
                const float* __restrict__ maskp,
                unsigned short* __restrict__ O, int Bsz, int SQa, int SKVa,
                int H, int HKV, float scale, long bstr_q, long tstr_q,
                long bstr_k, long tstr_k,
                const int* __restrict__ cu = nullptr,
                const int* __restrict__ blk_seq = nullptr,
                const int* __restrict__ blk_qb = nullptr,
                const int* __restrict__ cu_k = nullptr, int window = 0,
                const unsigned short* __restrict__ Kr = nullptr,
                const float* __restrict__ sink = nullptr,
                const unsigned short* __restrict__ gate = nullptr,
                int ld_gate = 0, const float* __restrict__ cs = nullptr,
                const float* __restrict__ sn = nullptr,
                const int* __restrict__ pos = nullptr) {
  constexpr int NWAVE = 4;  // waves per workgroup (8 measured slower)
  constexpr int QBLK = NWAVE * QWAVE;       // q rows per workgroup
  constexpr int NCH = D / 8;             // 16B chunks per K row
  constexpr int NCHV = DV / 8;           // 16B chunks per V row
  constexpr int DBLK = DV / 32;          // 32-wide d blocks of V
  constexpr int KTILE_B = KVBLK * D * 2; // K tile bytes
  constexpr int RTILE_B = KVBLK * ROT * 2; // shared key part of a tile
  constexpr int VTILE_B = KVBLK * DV * 2;  // V tile bytes

  const int lane = threadIdx.x & 63;
  // A wave number that the compiler knows to be uniform, and copies that it
  // does not know of (copy_to_lds), take fewer registers: packed proteins, 20
  // heads of 64, 108.5 -> 104 us. Heads of 128 are ordered worse with the
  // first: 4 x 4096 causal 655 against 692.
  const int wid = D + DV <= 192
                      ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)
                      : threadIdx.x >> 6;
  const int h = lane >> 5;   // half index within wave
  const int qcol = lane & 31;

  int qb, b, head;
  if (VARLEN) {
    const int nblk = WINDOW ? gridDim.x / H : SQa;
    if (!WINDOW && (int)blockIdx.x >= nblk * H) {
      const long n8 = (long)H * DV / 8;
      const long first = (long)cu[Bsz] * n8, end = (long)SKVa * n8;
      const long step = (gridDim.x - nblk * H) * blockDim.x;
      for (long i = first + (long)(blockIdx.x - nblk * H) * blockDim.x +
                    threadIdx.x;
           i < end; i += step)
        reinterpret_cast<i32x4*>(O)[i] = i32x4{0, 0, 0, 0};
      return;
    }
    // neighbouring q-blocks of one head share most of their keys: give
    // each XCD a contiguous run of them
    const int bid = xcd_run(blockIdx.x, nblk * H);
    head = bid / nblk;
    const int i = bid % nblk;
    b = blk_seq[i];
    qb = blk_qb[i];
  } else {
    const int nqb0 = (SQa + QBLK - 1) / QBLK;
    // keep the q-blocks sharing one (b, head)'s K/V on one XCD's L2
    // (+12% at D=128/GQA).
    const int bid = xcd_run(blockIdx.x, Bsz * H * nqb0);
    // causal: the blocks with most keys first, they would be the tail
    qb = CAUSAL ? nqb0 - 1 - bid % nqb0 : bid % nqb0;
    const int bh = bid / nqb0;
    head = bh % H;
    b = bh / H;
  }
  const int SQ = VARLEN ? cu[b + 1] - cu[b] : SQa;
  const int SKV = WINDOW ? cu_k[b + 1] - cu_k[b] : VARLEN ? SQ : SKVa;
  const int shift = WINDOW ? SKV - SQ : 0;  // key index of query 0
  const int kvhead = head / (H / HKV);

  const long ostride = (long)H * DV;
  const long qbase = VARLEN ? (long)cu[b] * tstr_q : (long)b * bstr_q;
  const long kbase = WINDOW   ? (long)cu_k[b] * tstr_k
                     : VARLEN ? (long)cu[b] * tstr_k
                              : (long)b * bstr_k;
  const unsigned short* Qb = Q + qbase + (long)head * (D + ROT);
  const unsigned short* Kb = Kt + kbase + (long)kvhead * D;
  const unsigned short* Vb = Vt + kbase + (long)kvhead * DV;
  unsigned short* Ob = O + (VARLEN ? (long)cu[b] : (long)b * SQ) * ostride +
                       (long)head * DV;

  const int q0w = qb * QBLK + wid * QWAVE;
  const int qrow_abs = q0w + qcol;
  const int qpos = qrow_abs + shift;
  const int qlo = WINDOW && qpos >= window ? qpos - window + 1 : 0;
  const int qload = qrow_abs < SQ ? qrow_abs : (SQ > 0 ? SQ - 1 : 0);

  const int offK[2] = {0, KTILE_B};
  constexpr int offR = 2 * KTILE_B;
  const int offV[2] = {offR + 2 * RTILE_B, offR + 2 * RTILE_B + VTILE_B};
  constexpr int offM = offR + 2 * RTILE_B + 2 * VTILE_B;
  const float* mask_lds = reinterpret_cast<const float*>(smem + offM);

  // the maximum is taken before scaling: with a negative scale, of the
  // negated scores
  const float scale2 = fabsf(scale) * LOG2E;
  const unsigned int flip = scale < 0.f ? 0x80008000u : 0u;

  int ntile = (SKV + KVBLK - 1) / KVBLK;
  if (CAUSAL) {
    const int qmax_blk = min(qb * QBLK + QBLK - 1, SQ - 1);
    ntile = min(ntile, (qmax_blk + shift) / KVBLK + 1);
  }
  unsigned long long some = 0;  // of the first 64 tiles
  auto holed = [&](int t) { return t >= 64 || (some >> t & 1); };
  auto mask_read = [&](int t) {
    return CAUSAL || holed(t) || (t + 1) * KVBLK > SKV;
  };

  // ---- Q fragments in registers ---------------------------------------
  bf16x8 qf[(D + ROT) / 16];
#pragma unroll
  for (int s = 0; s < (D + ROT) / 16; ++s) {
    frag_u f;
    f.v = *reinterpret_cast<const bf16x8*>(Qb + (long)qload * tstr_q +
                                           s * 16 + h * 8);
#pragma unroll
    for (int i = 0; i < 4; ++i) f.d[i] ^= flip;
    qf[s] = f.v;
  }
  float m = -1e30f, l = 0.f;
  f32x16 accO[DBLK];
#pragma unroll
  for (int d = 0; d < DBLK; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) accO[d][i] = 0.f;

  // ---- staging: 1 KiB pieces of whole rows, swizzled source -------------
  // Where all rows of a tile exist, from pointers that the wave shares and at
  // offsets of the lanes that stay: the 64-bit products of an address for every
  // copy were a sixth of a tile's vector cycles at D = 64.
  const int swid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned int lds0 = (unsigned int)(uintptr_t)(
      const __attribute__((address_space(3))) char*)smem;
  const bool near = tstr_k < 1L << 24;  // offsets of 32 bits
  auto kpart = [&](int row) { return (lane % NCH) ^ (row & (NCH - 1)); };
  auto vpart = [&](int row) { return (lane % NCHV) ^ ((row & 3) << 1); };
  auto rpart = [&](int row) { return (lane & 7) ^ (row & 7); };
  constexpr int KROWS = 1024 / (2 * D), VROWS = 1024 / (2 * DV);
  unsigned int kat = (swid * KROWS + lane / NCH) * ((unsigned int)tstr_k * 2);
  unsigned int vat = (swid * VROWS + lane / NCHV) * ((unsigned int)tstr_k * 2);
  auto rows = [&](auto each, auto whole, const unsigned short* from, long ld,
                  unsigned int lane_at, auto part, int k0, int to) {
    constexpr int R = decltype(each)::value;  // rows of a piece
    const int row = swid * R + lane / (64 / R);
#pragma unroll
    for (int p = 0; p < KVBLK / R / NWAVE; ++p) {
      const int more = p * NWAVE * R, at = to + (p * NWAVE + swid) * 1024;
      if constexpr (decltype(whole)::value)
        copy_to_lds(from + (k0 + more) * ld, lane_at + part(row + more) * 16,
                    lds0 + at);
      else
        copy_to_lds(from + (long)min(k0 + row + more, SKV - 1) * ld +
                        part(row + more) * 8,
                    smem + at);
    }
  };
  auto stage = [&](int k0, int buf) {
    if (HAS_MASK && wid == 0 && (k0 == 0 || mask_read(k0 / KVBLK)))
      copy_to_lds<4>(maskp + (long)b * SKV + min(k0 + lane, SKV - 1),
                     smem + offM + buf * KVBLK * 4);
    auto copies = [&](auto whole) {
      rows(std::integral_constant<int, KROWS>{}, whole, Kb, tstr_k, kat, kpart,
           k0, offK[buf]);
      if constexpr (ROT > 0) {
        static_assert(ROT == 64, "eight 16-byte pieces per row");
        rows(std::integral_constant<int, 8>{}, whole, Kr + (long)cu_k[b] * ROT,
             ROT, (swid * 8 + lane / 8) * (ROT * 2), rpart, k0,
             offR + buf * RTILE_B);
      }
      rows(std::integral_constant<int, VROWS>{}, whole, Vb, tstr_k, vat, vpart,
           k0, offV[buf]);
    };
    if (near && k0 + KVBLK <= SKV) copies(std::true_type{});
    else copies(std::false_type{});
  };
  int tile0 = 0;  // first tile that any row of this workgroup sees
  if (WINDOW) {
    const int first = qb * QBLK + shift - window + 1;
    tile0 = first > 0 ? first / KVBLK : 0;
  }

  // V^T fragments: 16 lanes take 4 keys x 16 columns; a lane's address is
  // key (lane & 15) / 4 of them, columns 4 * (lane & 3)
  const int vi = lane & 15;
  int v_off[2];  // of column blocks 0 and 1 (of 32); others 128 bytes on
#pragma unroll
  for (int d = 0; d < 2; ++d)
    v_off[d] = (4 * h + (vi >> 2)) * (2 * DV) +
               ((d * 2 + ((lane >> 4) & 1)) ^ (vi >> 2)) * 32 + (vi & 3) * 8;

  if (tile0 < ntile) stage(tile0 * KVBLK, 0);
  // ---- mask: which tiles have a number at all, and where the last key lies
  // that is not -inf in log2 units: the weight of those behind it is 0, their
  // tiles are left out. 64 x 203 with a quarter of the keys masked, 12 heads
  // of 64, 33 -> 27 us; 16 x 1024, 32 heads of 128, causal, 264 -> 234; with
  // nothing masked 512 x 512 takes as long as when a flag was read per tile,
  // for what the tiles save the first look costs ---------------------------
  if constexpr (HAS_MASK) {
    const float* mrow = maskp + (long)b * SKV;
    int live = 0;
#pragma unroll 8
    for (int t = 0; t < ntile; ++t) {
      const int k = t * KVBLK + lane;
      const float v = mrow[min(k, SKV - 1)];
      if (__any(!(v * LOG2E == -INFINITY))) live = t + 1;
      if (t < 64 && __any(v != 0.f)) some |= 1ull << t;
    }
    ntile = live;
  }
  // (the first tile is on its way)
  if constexpr (!WINDOW)
    if (cs != nullptr && q0w < SQ) {
      const long row = (VARLEN ? (long)cu[b] : (long)b * SQ) + qload;
      const long at = (long)pos[row] * (D / 2) + h * 8;
#pragma unroll
      for (int s = 0; s < D / 32; ++s) {
        float co[8], si[8], x[8], y[8];
        load8(cs + at + s * 16, co);
        load8(sn + at + s * 16, si);
        bf8_to_f32(__builtin_bit_cast(s16x8, qf[s]), x);
        bf8_to_f32(__builtin_bit_cast(s16x8, qf[s + D / 32]), y);
        s16x8 a, e;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          a[i] = (short)f2bf(x[i] * co[i] - y[i] * si[i]);
          e[i] = (short)f2bf(y[i] * co[i] + x[i] * si[i]);
        }
        qf[s] = __builtin_bit_cast(bf16x8, a);
        qf[s + D / 32] = __builtin_bit_cast(bf16x8, e);
      }
    }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  int cur = 0;
  for (int t = tile0; t < ntile; ++t) {
    const int k0 = t * KVBLK;
    const bool have_next = t + 1 < ntile;
    if (have_next) stage(k0 + KVBLK, cur ^ 1);  // into the other buffer

    const bool wave_active =
        q0w < SQ && (!CAUSAL || k0 <= q0w + shift + QWAVE - 1) &&
        (!WINDOW || k0 + KVBLK - 1 > q0w + shift - window);

    if (wave_active) {
      // ---- QK^T: two 32-key blocks, side by side ------------------------
      f32x16 sc[2];
      const f32x16 zero = {};
#pragma unroll
      for (int s = 0; s < D / 16; ++s)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          const int key = kb * 32 + (lane & 31);
          const int swz = (s * 2 + h) ^ (key & (NCH - 1));
          const bf16x8 kf = *reinterpret_cast<const bf16x8*>(
              smem + offK[cur] + key * (2 * D) + swz * 16);
          sc[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              kf, qf[s], s == 0 ? zero : sc[kb], 0, 0, 0);
        }
#pragma unroll
      for (int s = 0; s < ROT / 16; ++s)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          const int key = kb * 32 + (lane & 31);
          const bf16x8 kf = *reinterpret_cast<const bf16x8*>(
              smem + offR + cur * RTILE_B + key * (2 * ROT) +
              (((s * 2 + h) ^ (key & 7)) * 16));
          sc[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              kf, qf[D / 16 + s], sc[kb], 0, 0, 0);
        }
      // ---- scores in log2 units; r of a block is key
      // (r & 3) + 8 (r >> 2) + 4 h ---------------------------------------
      bool masked;  // whether a row of the wave does not see a key
      if (WINDOW)
        masked = k0 + KVBLK - 1 > q0w + shift ||
                 k0 <= q0w + QWAVE - 1 + shift - window;
      else
        masked = k0 + KVBLK > SKV || (CAUSAL && k0 + KVBLK - 1 > q0w) ||
                 (HAS_MASK && holed(t));
      float pmax = -INFINITY, mul;
      if (masked) {
        const unsigned int wspan = WINDOW ? qpos - qlo : 0;
        const int woff = k0 + 4 * h - qlo;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            f32x4 mv = {0.f, 0.f, 0.f, 0.f};
            if (HAS_MASK)
              mv = *reinterpret_cast<const f32x4*>(
                  mask_lds + cur * KVBLK + kb * 32 + g * 8 + 4 * h);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const int e = kb * 32 + g * 8 + j;  // key - k0 - 4h
              float s2 = sc[kb][g * 4 + j] * scale2;
              if (HAS_MASK) s2 += mv[j] * LOG2E;
              // WINDOW: key k is visible when 0 <= k - qlo <= qpos - qlo,
              // one unsigned compare
              if (WINDOW)
                s2 = (unsigned int)(woff + e) <= wspan ? s2 : -INFINITY;
              else {
                if (CAUSAL && k0 + 4 * h + e > qrow_abs) s2 = -INFINITY;
                if (k0 + 4 * h + e >= SKV) s2 = -INFINITY;
              }
              sc[kb][g * 4 + j] = s2;
              pmax = fmaxf(pmax, s2);
            }
          }
        mul = 1.f;
      } else {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r) pmax = fmaxf(pmax, sc[kb][r]);
        pmax *= scale2;
        mul = scale2;
      }
      pmax = lanes_max<32>(pmax);
      // defer-max (THR=8 in log2 units): skip the O rescale while the
      // running max has not grown by more than THR — P is then bounded by
      // 2^THR, which the fp32 l/O accumulation absorbs. The decision covers
      // THIS tile's P entirely (nothing of this tile is exponentiated
      // before the decision).
      float alpha = 1.f;
      if (!__all(pmax - m <= 8.f)) {
        const float mn = fmaxf(fmaxf(m, pmax), -1e30f);
        alpha = __builtin_amdgcn_exp2f(m - mn);
        m = mn;
#pragma unroll
        for (int d = 0; d < DBLK; ++d)
#pragma unroll
          for (int i = 0; i < 16; ++i) accO[d][i] *= alpha;
      }
      float rs[4];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float e = __builtin_amdgcn_exp2f(fmaf(sc[kb][r], mul, -m));
          sc[kb][r] = e;
          rs[r & 3] = kb * 16 + r < 4 ? e : rs[r & 3] + e;
        }
      // (kept apart to the end, the sums of both lane halves are rounded
      // otherwise, and so are some outputs; the swap of every tile is 0 to 1%:
      // 512 x 512 of 12 heads of 64 547 -> 553 us, 4 x 4096 of 32 of 128 592, 594)
      l = fmaf(l, alpha, lanes_sum<32>((rs[0] + rs[1]) + (rs[2] + rs[3])));

      // ---- PV, 16 keys at a time --------------------------------------
#pragma unroll
      for (int kh = 0; kh < 4; ++kh) {
        frag_u pa;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          pa.d[i] = pack_bf16(sc[kh >> 1][(kh & 1) * 8 + i * 2],
                              sc[kh >> 1][(kh & 1) * 8 + i * 2 + 1]);
#pragma unroll
        for (int d = 0; d < DBLK; ++d) {
          frag_u vf;
          const char* src = smem + offV[cur] + v_off[d & 1] + (d >> 1) * 128 +
                            kh * 16 * (2 * DV);
#pragma unroll
          for (int j = 0; j < 2; ++j)
            vf.h[j] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) s16x4*)(
                    src + j * 8 * (2 * DV)));
          accO[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              vf.v, pa.v, accO[d], 0, 0, 0);
        }
      }
    }

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();  // ONE barrier per tile
    cur ^= 1;
  }

  // ---- epilogue: a swap of lane halves leaves 8 columns on each ---------
  float inv_l = (l > 0.f) ? 1.f / l : 0.f;
  if (WINDOW && sink != nullptr && l > 0.f) {
    const float s = sink[head] * LOG2E, top = fmaxf(m, s);
    const float a = __builtin_amdgcn_exp2f(m - top);
    inv_l = a / (l * a + __builtin_amdgcn_exp2f(s - top));
  }
  if (WINDOW && gate != nullptr)
    inv_l *= sigmoid_exact(bf2f(gate[(cu[b] + (long)qload) * ld_gate + head]));
#pragma unroll
  for (int d = 0; d < DBLK; ++d)
#pragma unroll
    for (int g = 0; g < 4; g += 2) {
      unsigned int w[2][2];
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          w[e][i] = pack_bf16(accO[d][(g + e) * 4 + i * 2] * inv_l,
                              accO[d][(g + e) * 4 + i * 2 + 1] * inv_l);
      const i32x2 s0 = __builtin_amdgcn_permlane32_swap((int)w[0][0],
                                                        (int)w[1][0], false,
                                                        false);
      const i32x2 s1 = __builtin_amdgcn_permlane32_swap((int)w[0][1],
                                                        (int)w[1][1], false,
                                                        false);
      if (qrow_abs < SQ)
        *reinterpret_cast<i32x4*>(Ob + (long)qrow_abs * ostride + d * 32 +
                                  g * 8 + h * 8) =
            i32x4{s0[0], s1[0], s0[1], s1[1]};
    }
}
