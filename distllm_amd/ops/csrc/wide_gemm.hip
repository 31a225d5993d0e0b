// Products of many rows: out[M,N] = x[M,K] @ W[N,K]^T with bias and
// activation or gated unit in the launch (the projections of encoder layers,
// prompts and step batches; reference distllm/embed/encoders/auto.py encode(),
// distllm/generate/generators/vllm_backend.py).
//
// A workgroup stays on its CU and makes one tile of 32 FM x 256 after the
// other, 4 waves (one per SIMD) with 16 FM x 128 each: the sums are all 256
// accumulation registers at FM = 8, and an operand byte read from LDS feeds
// twice the matrix work of a 128 x 64 wave tile. K goes by stages of 64 columns
// through a ring of five LDS slots of 32 KiB, one for a stage of x or of W
// (all 160 KiB): x is copied three stages ahead, W two, over the edges of
// tiles, so that no tile begins with a wait. A stage has two halves of 32
// columns; while the matrix cores work on the fragments of one, those of the
// next are read and the copies of later stages started, at most one of either
// behind a product, in the shadow of its 16 cycles. One barrier per stage.
//
// W's rows are dealt to the fragments so that a lane's eight sums of a row are
// eight neighbouring columns: the tile leaves the registers in whole lines,
// without LDS. The stores drain during the next tile: vmcnt counts in order,
// and all that the next stage waits for is older than they are.
//
// Bounds, measured: dense products draw the card's full power (1.6 to 1.7 GHz
// at 78% of the matrix cores' cycles; with zeros as inputs the same launch is
// 1.2 to 1.3 times as fast), copies are what they wait for else.
#include <type_traits>

#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef unsigned short u16;

extern __shared__ __attribute__((aligned(16))) char smem[];

enum WgAct { WG_NONE = 0, WG_GELU_TANH = 1, WG_GELU_ERF = 2, WG_SILU = 3,
             WG_SWIGLU = 4, WG_CLAMPED = 5 };

struct WgArgs {
  const u16 *X, *W, *bias;
  u16* out;
  int M, N, K;  // of the product; gated units have N / 2 columns of output
  float limit, alpha, shift;
  unsigned by_span, by_last;  // 2^32 over the divisor, rounded up
};

constexpr int WG_SLOT = 32768;
constexpr int WG_GROUP = 8;  // row tiles that go over the columns together

// x Phi(x) in 32 bits. Phi(-|x|) is 2 to a polynomial of |x| of degree 7 that is
// -1 at 0 and falls everywhere, fitted with the least largest error of Phi, below
// 2e-7 or 3e-5 of it. Against 64 bits, and gelu_erf (erf by a reciprocal and an
// exponential, 22 issue slots where this takes 14): largest error 2.7e-7 (4.7e-7); of
// results above 0.01 1.9e-6 of them (1.6e-5), above 1e-4 3.4e-4 (1.1e-3); for |x|
// below 1e-3 1.4e-7 (3.5e-7). Degree 5 leaves 6.7e-7, 5.2e-5, 4.2e-3 and 4.3e-6, at
// -3.5 and below as much as the rounding to 16 bits; us, degree 5 and 7: 262144 x
// 3072 x 768 1217, 1250; 12992 x 3072 x 768 69.6, 72.5; 16384 x 5120 x 1280 183.5,
// 186.6. Degree 6 cannot fall everywhere and be closer than 5.
__device__ __forceinline__ float wg_gelu(float x) {
  const float y = fabsf(x);
  float p = fmaf(y, -7.365080705312721e-07f, 4.1180137486662716e-05f);
  p = fmaf(p, y, -0.000798956782091409f);
  p = fmaf(p, y, 0.008115779608488083f);
  p = fmaf(p, y, -0.05338641256093979f);
  p = fmaf(p, y, -0.4588525891304016f);
  p = fmaf(p, y, -1.1511530876159668f);
  p = fmaf(p, y, -1.f);
  // infinity times zero is kept out of a positive x; minus infinity gives NaN,
  // as x Phi(x) written down does, and NaN is in p
  return fmaf(-fabsf(fminf(x, 3e38f)), __builtin_amdgcn_exp2f(p),
              fmaxf(x, 0.f));
}

template <int ACT>
__device__ __forceinline__ float wg_act(float v) {
  if (ACT == WG_GELU_TANH) return fast_gelu(v);
  if (ACT == WG_GELU_ERF) return wg_gelu(v);
  if (ACT == WG_SILU) return silu(v);
  return v;
}

// A buffer of raw bytes: reads behind its end are zeros, stores are dropped.
__device__ __forceinline__ i32x4 wg_buffer(const void* p, long bytes) {
  const unsigned long a = (unsigned long)p;
  i32x4 r;
  r[0] = __builtin_amdgcn_readfirstlane((int)a);
  r[1] = __builtin_amdgcn_readfirstlane((int)(a >> 32) & 0xffff);
  r[2] = __builtin_amdgcn_readfirstlane(
      (int)(unsigned)(bytes < 0xfffffff0L ? bytes : 0xfffffff0L));
  r[3] = 0x00020000;
  return r;
}

// 16 bytes a lane to LDS, in order of the lanes from byte base + add (a
// constant) on. In assembly, so that the compiler waits for none of them (see
// copy_to_lds), and in two parts, between which a wait state has to pass and no
// other copy may come: a product in the loop (1 to 1.5% faster than a nop).
__device__ __forceinline__ void wg_copy_to(int base, int add) {
  asm volatile("s_add_u32 m0, %0, %1" : : "s"(base), "i"(add) : "scc");
}
__device__ __forceinline__ void wg_copy(const i32x4& buf, int lane_at,
                                        int at) {
  asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds"
               :
               : "v"(lane_at), "s"(buf), "s"(at)
               : "memory");
}

template <int N>
__device__ __forceinline__ void wg_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}

// slot offset `at` + n slots, round the ring of five
__device__ __forceinline__ int wg_round(int at, int n) {
  at += n * WG_SLOT;
  return at >= 5 * WG_SLOT ? at - 5 * WG_SLOT : at;
}

template <int ACT, int FM, bool STREAM>
__global__ void __launch_bounds__(256, 1) wide_gemm_kernel(const WgArgs p) {
  constexpr bool GLU = ACT >= WG_SWIGLU;
  constexpr int BM = FM * 32;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int mh = wid >> 1, nh = wid & 1;  // the wave's half of rows, columns
  const int ntm = (p.M + BM - 1) / BM, ntn = p.N / 256;

  // every XCD has a run of tiles of its own, its workgroups take turns
  const int tiles = ntm * ntn, per = gridDim.x >> 3;
  const int xcd = blockIdx.x & 7;
  const int t0 = (int)((long)tiles * xcd / 8) + (blockIdx.x >> 3);
  const int t1 = (int)((long)tiles * (xcd + 1) / 8);
  if (t0 >= t1) return;
  // WG_GROUP row tiles go over the columns together: 32 workgroups then read
  // 8 and 4 panels rather than 1 and 32 (16384 x 28672 x 4096: 2690 us in
  // plain order, 2460)
  auto where = [&](int t, int& tm, int& tn) {
    const int group = __umulhi((unsigned)t, p.by_span);
    const int rem = t - group * (WG_GROUP * ntn), tm0 = group * WG_GROUP;
    const bool full = tm0 + WG_GROUP <= ntm;
    const int rows = full ? WG_GROUP : ntm - tm0;
    tn = full        ? rem / WG_GROUP
         : rows == 1 ? rem
                     : (int)__umulhi((unsigned)rem, p.by_last);
    tm = tm0 + rem - tn * rows;
  };

  // ---- copies: rows of 128 bytes whose 16-byte pieces are XOR-ed with the row
  const int ldb = p.K * 2;
  const int lrow = lane >> 3, piece = ((lane & 7) ^ lrow) * 16;
  i32x4 xbuf, wbuf;
  int xlane[FM], wlane[8];
  int xt = t0, wt = t0, xk = 0, wk = 0;  // tile, byte in a row: what is next
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    // row j of fragment f of a half of the columns
    const int half = (wid * 8 + i) >> 4, f = ((wid * 8 + i) >> 1) & 7;
    const int j = (i & 1) * 8 + lrow;
    wlane[i] = (GLU ? (f >> 2) * (p.N / 2) + half * 64 + j * 4 + (f & 3)
                    : half * 128 + j * 8 + f) *
                   ldb + piece;
  }
  auto x_tile = [&]() {
    int tm, tn;
    where(xt, tm, tn);
    const int rows = min(BM, p.M - tm * BM);
    xbuf = wg_buffer(p.X + (long)tm * BM * p.K, (long)rows * ldb);
    int row = wid * (FM * 8) + lrow;
    asm volatile("" : "+v"(row));  // not kept in registers for every piece
#pragma unroll
    for (int i = 0; i < FM; ++i)
      xlane[i] = __umul24(min(row + i * 8, rows - 1), ldb) + piece;
  };
  auto w_tile = [&]() {
    int tm, tn;
    where(wt, tm, tn);
    const int n0 = tn * (GLU ? 128 : 256);
    wbuf = wg_buffer(p.W + (long)n0 * p.K, (long)(p.N - n0) * ldb);
  };
  // behind the last tile it is copied again, into slots that nothing reads
  auto x_next = [&]() {
    xk += 128;
    if (xk == ldb) {
      xk = 0;
      if (xt + per < t1) xt += per;
      x_tile();
    }
  };
  auto w_next = [&]() {
    wk += 128;
    if (wk == ldb) {
      wk = 0;
      if (wt + per < t1) wt += per;
      w_tile();
    }
  };
  x_tile();
  w_tile();
  int fill = 0;  // slot of the next copies: x, W, x, W, ...
  auto x_to = [&](int i) { wg_copy_to(fill + wid * (FM * 1024), i * 1024); };
  auto w_to = [&](int i) { wg_copy_to(fill + wid * 8192, i * 1024); };
  auto x_copy = [&](int i) { wg_copy(xbuf, xlane[i], xk); };
  auto w_copy = [&](int i) { wg_copy(wbuf, wlane[i], wk); };
#pragma unroll
  for (int s = 0; s < 2; ++s) {
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      x_to(i);
      asm volatile("s_nop 0");
      x_copy(i);
    }
    x_next();
    fill = wg_round(fill, 1);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      w_to(i);
      asm volatile("s_nop 0");
      w_copy(i);
    }
    w_next();
    fill = wg_round(fill, 1);
  }

  // ---- fragments: 16 rows x 32 columns
  const int xrow = mh * (FM * 2048) + r * 128, wrow = nh * 16384 + r * 128;
  const int col0 = (g ^ (r & 7)) * 16, col1 = col0 ^ 64;  // of either half
  int xs = 0, ws = WG_SLOT;  // slots of the stage that is read
  bf16x8 x0[FM], w0[8], x1[FM], w1[8];
  f32x4 acc[FM][8];
#pragma unroll
  for (int i = 0; i < FM * 8; ++i) acc[i >> 3][i & 7] = {0.f, 0.f, 0.f, 0.f};
  wg_wait<FM + 8>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < 8; ++i)
    w0[i] = *reinterpret_cast<const bf16x8*>(smem + ws + wrow + col0 + i * 2048);
#pragma unroll
  for (int i = 0; i < FM; ++i)
    x0[i] = *reinterpret_cast<const bf16x8*>(smem + xs + xrow + col0 + i * 2048);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");

  // The products of one half; behind them one by one the reads of the next
  // half and, COPY, the copies of x (1) or W (2). START: the sums begin here,
  // in assembly because the compiler would keep them elsewhere and move them.
  constexpr int READS = FM + 8, EVERY = (FM * 8 - 10) / READS;
  auto half = [&](auto start, auto copies_x, const char* xp, const char* wp,
                  bf16x8(&xa)[FM], bf16x8(&wa)[8], bf16x8(&xn)[FM],
                  bf16x8(&wn)[8]) {
    constexpr bool START = decltype(start)::value;
    constexpr bool CX = decltype(copies_x)::value;
    constexpr int GAP = FM > 4 ? 4 : 3, N = CX ? FM : 8;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < FM * 8; ++s) {
      f32x4& c = acc[s >> 3][s & 7];
      if constexpr (START)
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0"
                     : "+a"(c)
                     : "v"(xa[s >> 3]), "v"(wa[s & 7]));
      else
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[s >> 3], wa[s & 7], c,
                                                    0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (s % EVERY == EVERY / 2 && s / EVERY < READS) {
        const int i = s / EVERY;
        if (i < 8)
          wn[i] = *reinterpret_cast<const bf16x8*>(wp + i * 2048);
        else
          xn[i - 8] = *reinterpret_cast<const bf16x8*>(xp + (i - 8) * 2048);
      }
      if (s % GAP == 1 && s / GAP < N) {
        if constexpr (CX) x_copy(s / GAP);
        else w_copy(s / GAP);
      }
      if (s % GAP == 0 && s / GAP < N) {
        if constexpr (CX) x_to(s / GAP);
        else w_to(s / GAP);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // all that was read of a slot is here before the barrier behind which it
    // is filled again
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  using Yes = std::true_type;
  using No = std::false_type;
  auto first = [&](auto start) {
    half(start, Yes{}, smem + xs + xrow + col1, smem + ws + wrow + col1, x0,
         w0, x1, w1);
    x_next();
    fill = wg_round(fill, 1);
    xs = wg_round(xs, 2);
    ws = wg_round(ws, 2);
  };
  auto second = [&]() {  // behind a wait for the next stage
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    half(No{}, No{}, smem + xs + xrow + col0, smem + ws + wrow + col0, x1, w1,
         x0, w0);
    w_next();
    fill = wg_round(fill, 1);
  };

  // Younger than the next stage are the copies of x of the one after it and, in
  // a later tile's first stage, the 4 FM stores of the tile before.
  bool later = false;
  for (int t = t0; t < t1; t += per) {
    first(Yes{});
    if (later) wg_wait<5 * FM>();
    else wg_wait<FM>();
    second();
    for (int k = 64; k < p.K; k += 64) {
      first(No{});
      wg_wait<FM>();
      second();
    }
    later = true;

    int tm, tn;
    where(t, tm, tn);
    int cols = GLU ? p.N / 2 : p.N;
    asm volatile("" : "+s"(cols));  // offsets are not kept over the loop
    const int rows = min(BM, p.M - tm * BM);
    const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(
        p.out + (long)tm * BM * cols, 0, rows * cols * 2, 0x00020000);
    const int n = tn * (GLU ? 128 : 256) + nh * (GLU ? 64 : 128) +
                  r * (GLU ? 4 : 8);
    float b[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) b[i] = 0.f;
    if (p.bias != nullptr) {
      if constexpr (GLU) {
        const s16x4 lo = *reinterpret_cast<const s16x4*>(p.bias + n);
        const s16x4 hi = *reinterpret_cast<const s16x4*>(p.bias + cols + n);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          b[i] = bf2f((u16)lo[i]);
          b[4 + i] = bf2f((u16)hi[i]);
        }
      } else {
        bf8_to_f32(*reinterpret_cast<const s16x8*>(p.bias + n), b);
      }
    }
    const int at = ((mh * (FM * 16) + g * 4) * cols + n) * 2;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      __builtin_amdgcn_sched_barrier(0);
      // the sums leave the accumulation registers here and not before
#pragma unroll
      for (int f = 0; f < 8; ++f) asm volatile("" : "+a"(acc[i][f]));
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int off = at + (i * 16 + q) * cols * 2;
        u16 o[8];
        if constexpr (GLU) {
#pragma unroll
          for (int f = 0; f < 4; ++f) {
            const float a = acc[i][f][q] + b[f], u = acc[i][4 + f][q] + b[4 + f];
            o[f] = f2bf(ACT == WG_SWIGLU ? silu(a) * u
                                         : clamped_glu(a, u, p.limit, p.alpha,
                                                       p.shift));
          }
          __builtin_amdgcn_raw_buffer_store_b64(
              *reinterpret_cast<const i32x2*>(o), out, off, 0, STREAM ? 2 : 0);
        } else {
#pragma unroll
          for (int f = 0; f < 8; ++f) o[f] = f2bf(wg_act<ACT>(acc[i][f][q] + b[f]));
          __builtin_amdgcn_raw_buffer_store_b128(
              *reinterpret_cast<const i32x4*>(o), out, off, 0, STREAM ? 2 : 0);
        }
      }
    }
  }
  // nothing is in flight to LDS that the next workgroup may have
  wg_wait<0>();
}

// Rows of a tile / 32: those with the least rounds of the card's 256 CUs times
// what a tile costs, which is its rows and, for W and the turn to the next tile, as
// much as 192 more. us, fm 8 to 4: 12992 x 768 x 768 19.8, 18.7, 17.9, 17.3, 22.6, by
// this rule 14, 13, 12, 11, 20; 8448 x 4096 x 14336 850, 794, 749, 894, 1004: 42, 39,
// 36, 44, 50. A round of 28672 x 4096 gated 80, 73, 68, 65, 62. Ties go to the larger
// tile. *tiles: their number.
static int wg_tile(int M, int N, long* tiles) {
  int best = 8;
  long least = -1;
  for (int fm = 8; fm >= 4; --fm) {
    const long n = (long)((M + 32 * fm - 1) / (32 * fm)) * (N / 256);
    const long cost = ((n + 7) / 8 + 31) / 32 * (fm + 6);
    if (least >= 0 && cost >= least) continue;
    least = cost;
    best = fm;
    *tiles = n;
  }
  return best;
}

// The tile with which this product is the faster one, 0 where another is.
// Measured against the library's product (and the activation's or unit's own
// launch), own time over its, in a graph, over weights that come from memory:
// - A single round, by the share of the card's 256 tiles of 256 rows that its tiles
//   make: without activation and K of 1536 and more 0.58 to 0.9 0.75 to 1.02, 0.5 to
//   0.55 1.04 to 1.08, below 1.1 to 1.9; a gated unit of K from 4096 on 0.54 and more
//   0.83 to 1.0, 0.44 1.02 to 1.23; with either and K of 1536 to 2048 0.43 and more
//   0.75 to 1.03, 0.38 1.0 to 1.09, 0.19 to 0.31 1.07 to 1.39. Shorter sums: without
//   activation 216 tiles and more 0.52 to 1.03, 120 to 192 0.67 to 1.24, fewer up to
//   1.55; with one, K to 1024, 96 tiles and more 0.5 to 1.09, K of 1280 to 1472 96 to
//   160 tiles 1.05 to 1.36, 176 to 192 0.95 to 1.1, more below that. Those 96 to 192
//   are taken for the host, which two or three calls cost 21 to 30 us and this one 6:
//   issued one after the other 0.78 to 1.0 (K of 1536 0.98 to 1.1), and an encoder
//   of 650 M weights on 700 to 1300 tokens 4840 and 4120 us.
// - Several rounds that fill less than half of the card without an activation: K of
//   1024 and more 1.08 to 1.1.
// - Long sums whose 256 x 256 tiles fill their rounds, which is the library's
//   best case: K of 1536 and more, a share of 0.87 and more 1.01 to 1.09, below
//   0.73 to 0.99. With K to 1280 0.86 to 1.0 all the same, and with an
//   activation or a unit 0.79 to 0.93 at any K.
extern "C" int wide_gemm_tile(int M, int N, int K, int act) {
  if (M <= 0 || N <= 0 || N % 256 || K % 64 || K < 128 ||
      (long)N * K >= 1L << 30 || M >= 1 << 30)
    return 0;
  long tiles = 0;
  const int fm = wg_tile(M, N, &tiles);
  const long ntn = N / 256;
  if (tiles * ntn * WG_GROUP >= 1L << 32)
    return 0;  // divisions by multiplication
  const long filled = tiles * fm;  // 2048 are a round of 256 tiles of 256 rows
  if (tiles <= 256) {
    if (K < 1536) {
      if (tiles < (act != WG_NONE ? 96 : 208)) return 0;
    } else if (filled <
               (act == WG_NONE ? 0.58f : K <= 2048 ? 0.43f : 0.5f) * 2048) {
      return 0;
    }
  } else if (act == WG_NONE && K >= 1024 &&
             filled < ((tiles + 7) / 8 + 31) / 32 * 1024) {
    return 0;
  }
  if (act == WG_NONE && K >= 1536) {
    const long most = (long)((M + 255) / 256) * ntn;
    if (most >= 0.87f * ((most + 255) / 256 * 256)) return 0;
  }
  return fm;
}

// fm: rows of a tile / 32, 4 to 8. K % 64 == 0 and at least 128, N % 256 == 0;
// act 4 and 5 are gated units.
extern "C" void launch_wide_gemm(const void* X, const void* W,
                                 const void* bias, void* out, int M, int N,
                                 int K, int act, float limit, float alpha,
                                 float shift, int fm, hipStream_t stream) {
  const int ntm = (M + 32 * fm - 1) / (32 * fm), ntn = N / 256;
  auto over = [](unsigned d) {
    return d > 1 ? (unsigned)(((1ul << 32) + d - 1) / d) : 0u;
  };
  const WgArgs a = {(const u16*)X, (const u16*)W, (const u16*)bias, (u16*)out,
                    M, N, K, limit, alpha, shift, over(WG_GROUP * ntn),
                    over(ntm % WG_GROUP)};
  // Results that the 256 MiB cache beside the memory cannot keep for the next
  // kernel go past it (262144 x 2304 x 768: 762 us kept, 738 past it; 12992 x
  // 3072 x 768 58.5 and 59.7).
  const bool past = (long)M * (act >= WG_SWIGLU ? N / 2 : N) * 2 > 256L << 20;
#define WG_LAUNCH(A, F, S)                                                  \
  hipLaunchKernelGGL((wide_gemm_kernel<A, F, S>), dim3(256), dim3(256),     \
                     5 * WG_SLOT, stream, a)
#define WG_ROWS(A)                            \
  case A:                                     \
    if (fm == 4) WG_LAUNCH(A, 4, false);      \
    else if (fm == 5) WG_LAUNCH(A, 5, false); \
    else if (fm == 6) WG_LAUNCH(A, 6, false); \
    else if (fm == 7) WG_LAUNCH(A, 7, false); \
    else if (past) WG_LAUNCH(A, 8, true);     \
    else WG_LAUNCH(A, 8, false);              \
    break
  switch (act) {
    WG_ROWS(0); WG_ROWS(1); WG_ROWS(2); WG_ROWS(3); WG_ROWS(4); WG_ROWS(5);
  }
#undef WG_ROWS
#undef WG_LAUNCH
}
