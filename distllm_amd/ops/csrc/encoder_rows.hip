// Products of an encoder's few rows (width H <= 1024) with what came ahead of
// them in launches of their own: the norm of a sum (launch_norm_rows, M <= 32 or
// 24) and the attention of short texts (launch_attn_rows, M <= 64). On so few rows
// a launch is latency: 2.9 us a norm, 4.8 the attention of 24 tokens, and the
// products 3 to 4. Here every workgroup norms, or attends, all rows again while
// its weights are on their way; 16 columns of W are a workgroup: 24 KiB of
// weights, and 74 KiB of rows to norm (24 x 768) or 110 KiB to attend, from L2.
// Twelve waves: a head each at 12 heads of 64, two rows each of 24.
//
// Sums, their order and all roundings are those of norm_fwd_small_kernel,
// attn_fwd_kernel and dg_ring_kernel, bit for bit: layers one by one go by
// these. So K is dealt to four waves in chunks of 64, and the other waves take
// other rows.
//
// What a launch is made of: the start of the waves, a round to L2 for the rows, the
// norm (vector units: every workgroup norms all rows) and the product. The weights
// are asked for ahead of all that and waited for behind it: as copies that the
// compiler cannot tell from accesses of LDS they were waited for ahead of the norm
// (24 rows, 2304 columns, under a profiler 5.5 us, now 4.9). 12 layers in a graph,
// us, norms in launches of their own and here: 768 on 4 rows 248 and 208, 16 259 and
// 217, 24 274 and 241, 32 317 and 296, 2 x 16 300 and 278; 1024 on 16 304 and 273,
// 24 332 and 309; 512 on 24 256 and 215.
#include "attention_kernel.h"
#include <algorithm>

typedef unsigned short u16;

namespace {

constexpr int NW = 12, COLS = 16, MSETS = NW / 4;

// x image in LDS: chunks of 64 numbers of MR rows (M in eights), whose 16-byte
// pieces are XOR-ed with the row. Tiles of 16 rows may read 8 past a chunk's
// end, of which nothing is kept.
__device__ __forceinline__ int piece_at(int row, int piece, int MR) {
  return ((piece >> 3) * MR + row) * 128 + ((piece & 7) ^ (row & 7)) * 16;
}
constexpr int up8(int n) { return (n + 7) / 8 * 8; }

__device__ __forceinline__ void lds_barrier() {
  // only LDS is waited for: loads and stores of memory go on
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// The workgroup's 16 rows of W, as chunks of 64 columns, by copies of 1 KiB.
// Straight-line code: a wave without a CP-th piece copies the last once more.
// KNOWN: to the compiler, so that waits for loads ahead of them do not wait for
// them, too; not where others are by copy_to_lds.
template <int CP, bool KNOWN>
__device__ __forceinline__ void start_weights(const u16* W, int H, char* ws) {
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane >> 3, lc = ((lane & 7) ^ lr) * 8;
  const u16* rows = W + (long)blockIdx.x * COLS * H;
  const __amdgpu_buffer_rsrc_t buffer = weight_rows(rows, COLS * H * 2);
#pragma unroll
  for (int i = 0; i < CP; ++i) {
    const int p = min(wid + i * NW, H / 32 - 1);
    const int at = (p & 1) * 8 * H + (p >> 1) * 64;
    if constexpr (KNOWN)
      copy_rows_to_lds(buffer, (lr * H + lc) * 2, at * 2, ws + p * 1024);
    else
      copy_to_lds(rows + at + lr * H + lc, ws + p * 1024);
  }
}

struct RowsEnd {
  const u16* bias;
  u16* out;
  int M, N;
};

// out[M, 16 columns] = act(x image @ (weights in LDS)^T + bias). All of the
// workgroup's waves; the images are whole and visible. act: of decode_gemm.
template <int ACT, int MT>
__device__ __forceinline__ void finish_product(const RowsEnd& e, int H,
                                               const char* xs, const char* ws,
                                               float* red, s16x4 bias) {
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4, MR = up8(e.M);
  constexpr int MINE = (MT + MSETS - 1) / MSETS;
  const int kw = wid & 3, first = wid >> 2;
  f32x4 acc[MINE];
#pragma unroll
  for (int j = 0; j < MINE; ++j) acc[j] = {0.f, 0.f, 0.f, 0.f};
  if (first < MT) {
    for (int c = kw; c < H / 64; c += 4)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const bf16x8 w = *reinterpret_cast<const bf16x8*>(
            ws + c * 2048 + r * 128 + (((h * 4 + g) ^ (r & 7)) * 16));
#pragma unroll
        for (int j = 0; j < MINE; ++j) {
          const int t = first + j * MSETS;
          if (t < MT)
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                w,
                *reinterpret_cast<const bf16x8*>(
                    xs + piece_at(t * 16 + r, c * 8 + h * 4 + g, MR)),
                acc[j], 0, 0, 0);
        }
      }
#pragma unroll
    for (int j = 0; j < MINE; ++j) {
      const int t = first + j * MSETS;
      if (t < MT)
        *reinterpret_cast<f32x4*>(red + ((kw * MT + t) * 64 + lane) * 4) =
            acc[j];
    }
  }
  lds_barrier();
  const int t = wid;
  const int m = t * 16 + r;
  if (t >= MT || m >= e.M) return;
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < 4; ++w)
    v += *reinterpret_cast<const f32x4*>(red + ((w * MT + t) * 64 + lane) * 4);
  s16x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = v[i] + bf2f((u16)bias[i]);
    if (ACT == 6) a = fast_gelu(a);
    if (ACT == 7) a = gelu_erf(a);
    o[i] = (short)f2bf(a);
  }
  *reinterpret_cast<s16x4*>(e.out + (long)m * e.N + blockIdx.x * COLS +
                            g * 4) = o;
}

__device__ __forceinline__ s16x4 load_bias(const RowsEnd& e) {
  return *reinterpret_cast<const s16x4*>(e.bias + blockIdx.x * COLS +
                                         ((threadIdx.x & 63) >> 4) * 4);
}

// Sum over 32 lanes, as wave_reduce_sum pairs them (16, 8, 4, 2, 1 apart).
__device__ __forceinline__ float half_reduce_sum(float v) {
  v = lanes_sum<16>(v);
  v += lane_turned<8>(v);
  v += lane_turned<4>(v);
  v += lane_turned<2>(v);
  v += lane_turned<1>(v);
  return v;
}

struct RowsNorm {
  const u16 *y, *res, *w, *b;
  u16* out;  // the normed rows, for the next sum
  float eps;
};

// ---- norm of y + res, then the product ---------------------------------------
// Half a wave has a row, 8 numbers a lane and up to NC times: numbers 256 k + 8
// lane. norm_fwd_small_kernel has them in waves of 512: the sums of k = 0, 1 and
// of 2, 3 meet after 32 lanes have been added up.
template <int ACT, int MT, int NC, int PASS>
__global__ void __launch_bounds__(NW * 64)
norm_rows_kernel(const RowsNorm n, const u16* __restrict__ W, int H,
                 const RowsEnd e) {
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31;
  char* xs = smem;
  const int MR = up8(e.M);
  char* ws = xs + MR * H * 2;
  float* red = reinterpret_cast<float*>(ws + 16 * H * 2);
  s16x8 yv[PASS][NC], rv[PASS][NC], wv[NC], bv[NC];
#pragma unroll
  for (int p = 0; p < PASS; ++p) {
    const long row =
        (long)min((p * NW + wid) * 2 + (lane >> 5), e.M - 1) * H;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const int c = min((k * 32 + l32) * 8, H - 8);
      yv[p][k] = *reinterpret_cast<const s16x8*>(n.y + row + c);
      rv[p][k] = *reinterpret_cast<const s16x8*>(n.res + row + c);
    }
  }
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const int c = min((k * 32 + l32) * 8, H - 8);
    wv[k] = *reinterpret_cast<const s16x8*>(n.w + c);
    bv[k] = *reinterpret_cast<const s16x8*>(n.b + c);
  }
  const s16x4 bias = load_bias(e);
  __builtin_amdgcn_sched_barrier(0);
  start_weights<NC == 3 ? 2 : 3, true>(W, H, ws);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int p = 0; p < PASS; ++p) {
    const int row = (p * NW + wid) * 2 + (lane >> 5);
    if ((p * NW + wid) * 2 >= e.M) break;
    float v[NC][8], s[2] = {0.f, 0.f}, q[2] = {0.f, 0.f};
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      float t[8], sum = 0.f, sumsq = 0.f;
      bf8_to_f32(yv[p][k], v[k]);
      bf8_to_f32(rv[p][k], t);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[k][i] += t[i];
        sum += v[k][i];
        sumsq += v[k][i] * v[k][i];
      }
      if ((k * 32 + l32) * 8 < H) {
        s[k >> 1] += sum;
        q[k >> 1] += sumsq;
      }
    }
    const float sum = half_reduce_sum(s[0]) + half_reduce_sum(s[1]);
    const float sumsq = half_reduce_sum(q[0]) + half_reduce_sum(q[1]);
    const float mean = sum / H;
    const float inv = rsqrtf(fmaxf(sumsq / H - mean * mean, 0.f) + n.eps);
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const int piece = k * 32 + l32;
      if (row < e.M && piece * 8 < H) {
        float wf[8], bf[8];
        bf8_to_f32(wv[k], wf);
        bf8_to_f32(bv[k], bf);
        s16x8 o;
#pragma unroll
        for (int i = 0; i < 8; ++i)
          o[i] = (short)f2bf((v[k][i] - mean) * inv * wf[i] + bf[i]);
        *reinterpret_cast<s16x8*>(xs + piece_at(row, piece, MR)) = o;
      }
    }
  }
  // (weights that came after the rows' numbers)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  lds_barrier();
  finish_product<ACT, MT>(e, H, xs, ws, red, bias);
  for (int row = blockIdx.x; row < e.M; row += gridDim.x)
    if ((int)threadIdx.x * 8 < H)
      *reinterpret_cast<s16x8*>(n.out + (long)row * H + threadIdx.x * 8) =
          *reinterpret_cast<const s16x8*>(xs + piece_at(row, threadIdx.x, MR));
}

// ---- attention of texts of up to 32 tokens, then the product ----------------
// A wave takes a text's head of 64 at a time: 32 queries against 32 keys, as
// attn_fwd_kernel with the one tile that there is; what it adds for keys past
// the text are zeros. Queries are copied to where their results will stand in
// the x image, keys and values beside them: whole lines, for the load path is
// what twelve waves share (queries and keys straight to the operands' registers
// and a mask number per key and lane: 6.1 us against 4.5 for 24 tokens).
constexpr int wave_lds(int S) { return up8(S) * 256 + 128; }

template <int MT, int CP>
__global__ void __launch_bounds__(NW * 64)
attn_rows_kernel(const u16* __restrict__ qkv, const float* __restrict__ mask,
                 const u16* __restrict__ W, int B, int S, int heads,
                 float scale, const RowsEnd e) {
  const int H = heads * 64, MR = up8(e.M), SR = up8(S);
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int q = lane & 31, h = lane >> 5, lr = lane >> 3;
  char* xs = smem;
  char* ws = xs + MR * H * 2;
  char* own = ws + 16 * H * 2;
  float* red = reinterpret_cast<float*>(own);  // when all have attended
  char* ks = own + wid * wave_lds(S);
  char* vs = ks + SR * 128;
  float* ms = reinterpret_cast<float*>(vs + SR * 128);
  const long ld = 3L * H;
  const int at = min(q, S - 1), units = B * heads;
  const float scale2 = scale * LOG2E;
  const s16x4 bias = load_bias(e);
  const int vi = lane & 15;
  int v_off[2];
#pragma unroll
  for (int d = 0; d < 2; ++d)
    v_off[d] = (4 * h + (vi >> 2)) * 128 +
               ((d * 2 + ((lane >> 4) & 1)) ^ (vi >> 2)) * 32 + (vi & 3) * 8;
  for (int u = wid; u < units; u += NW) {
    const int b = u / heads, head = u % heads;
    const u16* base = qkv + (long)b * S * ld + head * 64;
    char* qs = xs + (head * MR + b * S) * 128;
    // (by a copy, too: for a load the compiler would wait until nothing is in
    // flight, the weights among it)
    if (lane < 32) copy_to_lds<4>(mask + b * S + at, ms);
    for (int p = 0; p < SR / 8; ++p) {
      const int row = p * 8 + lr;
      const u16* src = base + min(row, S - 1) * ld;
      // other texts' rows follow
      if (row < S)
        copy_to_lds(src + ((lane & 7) ^ ((b * S + row) & 7)) * 8,
                    qs + p * 1024);
      copy_to_lds(src + H + ((lane & 7) ^ lr) * 8, ks + p * 1024);
      copy_to_lds(src + 2 * H + ((lane & 7) ^ ((row & 3) << 1)) * 8,
                  vs + p * 1024);
    }
    if (u == wid) {
      start_weights<CP, false>(W, H, ws);
      asm volatile("s_waitcnt vmcnt(%0)" ::"i"(CP) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    if (lane < 32) ms[lane] = q < S ? ms[lane] * LOG2E : -INFINITY;
    wave_sync();

    f32x16 sc = {};
#pragma unroll
    for (int s = 0; s < 4; ++s)
      sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          *reinterpret_cast<const bf16x8*>(ks + at * 128 +
                                           (((s * 2 + h) ^ (at & 7)) * 16)),
          *reinterpret_cast<const bf16x8*>(
              qs + at * 128 + (((s * 2 + h) ^ ((b * S + at) & 7)) * 16)),
          sc, 0, 0, 0);
    float top = -INFINITY;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 mv = *reinterpret_cast<const f32x4*>(ms + g * 8 + 4 * h);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        sc[g * 4 + j] = sc[g * 4 + j] * scale2 + mv[j];
        top = fmaxf(top, sc[g * 4 + j]);
      }
    }
    top = fmaxf(lanes_max<32>(top), -1e30f);
    float rs[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      sc[r] = __builtin_amdgcn_exp2f(sc[r] - top);
      rs[r & 3] += sc[r];
    }
    float l = (rs[0] + rs[1]) + (rs[2] + rs[3]);
    l = lanes_sum<32>(l);
    const float inv_l = l > 0.f ? 1.f / l : 0.f;

    f32x16 acc[2] = {};
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      frag_u pa;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        pa.d[i] = pack_bf16(sc[kh * 8 + i * 2], sc[kh * 8 + i * 2 + 1]);
      // keys from 8 on past the text have no row in LDS; their weights are 0
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        frag_u vf;
#pragma unroll
        for (int j = 0; j < 2; ++j)
          vf.h[j] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) s16x4*)(
                  vs + v_off[d] + min(kh * 2 + j, SR / 8 - 1) * 1024));
        acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf.v, pa.v, acc[d], 0,
                                                         0, 0);
      }
    }
    if (q < S) {
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const i32x2 o = {
              (int)pack_bf16(acc[d][g * 4] * inv_l, acc[d][g * 4 + 1] * inv_l),
              (int)pack_bf16(acc[d][g * 4 + 2] * inv_l,
                             acc[d][g * 4 + 3] * inv_l)};
          *reinterpret_cast<i32x2*>(
              xs + piece_at(b * S + q, head * 8 + d * 4 + g, MR) + h * 8) = o;
        }
    }
    // all is read before the next head is copied
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  // a wave that had no head has its weights to copy
  if (wid >= units) start_weights<CP, false>(W, H, ws);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  lds_barrier();
  finish_product<0, MT>(e, H, xs, ws, red, bias);
}

// S: of the attention, 0 without one
int rows_lds(int M, int H, int S) {
  const int sums = (M + 15) / 16 * 4096, own = S ? NW * wave_lds(S) : 0;
  return (up8(M) + 16) * H * 2 + std::max(sums, own);
}
constexpr int LDS_MOST = 160 * 1024;

}  // namespace

// Whether M rows of H numbers are normed by every workgroup. They fit up to 56
// rows of 1024, but every workgroup norms them all, and a launch of its own costs
// the same whatever they are. From 25 rows on a wave has a second pair of rows;
// 12 layers, own launches and joined, us: 24 rows of 512 256 and 215, 768 274 and
// 241, 832 289 and 270, 1024 332 and 309; 25 rows of 768 313 and 292, 32 317 and 296.
// Beyond, while the copies were waited for ahead of the norm: 25 rows of 832 334 and
// 337, 896 336 and 342, 1024 403 and 404; 32 rows of 832 339 and 346, 1024 415 and
// 419; 48 rows of 768 381 and 384, 64 rows 390 and 423.
extern "C" bool norm_rows_fit(int M, int H) {
  return M >= 1 && M <= (H <= 768 ? 32 : 24) && H % 64 == 0 && H >= 64 &&
         H <= 1024 && rows_lds(M, H, 0) <= LDS_MOST;
}

// Whether the attention fits the twelve waves in at most two turns, and LDS
// (texts of 25 to 32 tokens at 12 heads do not).
extern "C" bool attn_rows_fit(int B, int S, int heads, int D) {
  return D == 64 && S >= 1 && S <= 32 && B * S <= 64 && heads <= 16 &&
         B * heads <= 2 * NW && rows_lds(B * S, heads * 64, S) <= LDS_MOST;
}

// act: 0, or decode_gemm's code of a GELU
extern "C" void launch_norm_rows(const void* y, const void* res, const void* w,
                                 const void* b, void* normed, float eps,
                                 const void* W, const void* bias, void* out,
                                 int M, int N, int H, int act,
                                 hipStream_t stream) {
  const RowsNorm n = {(const u16*)y, (const u16*)res, (const u16*)w,
                      (const u16*)b, (u16*)normed, eps};
  const RowsEnd e = {(const u16*)bias, (u16*)out, M, N};
#define NR(A, MT, NC, P)                                                    \
  hipLaunchKernelGGL((norm_rows_kernel<A, MT, NC, P>), dim3(N / COLS),      \
                     dim3(NW * 64), rows_lds(M, H, 0), stream, n,       \
                     (const u16*)W, H, e)
#define NR_A(A)                                                             \
  do {                                                                      \
    if (H > 768 && M <= 16) NR(A, 1, 4, 1);                                 \
    else if (H > 768) NR(A, 2, 4, 1);                                       \
    else if (M <= 16) NR(A, 1, 3, 1);                                       \
    else if (M <= 24) NR(A, 2, 3, 1);                                       \
    else NR(A, 2, 3, 2);                                                    \
  } while (0)
  if (act == 6) NR_A(6);
  else if (act == 7) NR_A(7);
  else NR_A(0);
#undef NR_A
#undef NR
}

// qkv [B * S, 3 * heads * 64], mask [B, S] additive; out [B * S, N]
extern "C" void launch_attn_rows(const void* qkv, const float* mask,
                                 const void* W, const void* bias, void* out,
                                 int B, int S, int heads, int N, float scale,
                                 hipStream_t stream) {
  const int M = B * S, H = heads * 64;
  const RowsEnd e = {(const u16*)bias, (u16*)out, M, N};
#define AR(MT, CP)                                                          \
  hipLaunchKernelGGL((attn_rows_kernel<MT, CP>), dim3(N / COLS),            \
                     dim3(NW * 64), rows_lds(M, H, S), stream,           \
                     (const u16*)qkv, mask, (const u16*)W, B, S, heads,     \
                     scale, e)
#define AR_M(CP)                                                            \
  do {                                                                      \
    if (M <= 16) AR(1, CP);                                                 \
    else if (M <= 32) AR(2, CP);                                            \
    else if (M <= 48) AR(3, CP);                                            \
    else AR(4, CP);                                                         \
  } while (0)
  if (H <= 768) AR_M(2);
  else AR_M(3);
#undef AR_M
#undef AR
}
