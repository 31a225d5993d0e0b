// Torch bindings for the distllm-amd HIP kernel library (gfx950).
// Everything but the matrix products (ext_gemm.cpp) and the latent-
// attention decoder (ext_latent.cpp). The ops layer fails loudly on GPU
// if this extension is missing — no silent eager fallback.
// All kernels are hand-written CDNA4 HIP (see *.hip in this directory);
// this file only validates tensors and forwards device pointers.
#include <climits>
#include <cmath>
#include <cstring>
#include <limits>
#include <numeric>

#include "ahead.h"
#include "ext_common.h"

extern "C" {
void launch_norm_fwd(const void*, const void*, const void*, const void*,
                     void*, void*, int, int, float, bool, hipStream_t);
void launch_bias_gelu(const void*, const void*, void*, long, int, bool,
                      hipStream_t);
void launch_swiglu(const void*, const void*, void*, long, hipStream_t);
void launch_swiglu_packed(const void*, void*, long, int, hipStream_t);
void launch_bias_add(const void*, const void*, void*, long, int, hipStream_t);
void launch_mean_pool(const void*, const int*, float*, float*, int, int, int,
                      int, bool, hipStream_t);
int mean_pool_shares(int, int);
void launch_embed_layer_norm(const long*, const long*, const void*,
                             const void*, const void*, const void*,
                             const void*, void*, long, int, int, long, long,
                             float, const void*, int, float*, hipStream_t);
void launch_key_bias(const void*, float*, long, int, hipStream_t);
void launch_rope_inplace(void*, const float*, const float*, const int*, long,
                         long, int, int, hipStream_t);
void launch_last_token_pool(const void*, const int*, float*, int, int, int,
                            bool, bool, hipStream_t);
void launch_l2_normalize(const float*, float*, int, int, hipStream_t);
void launch_adjacent_cosine(const float*, float*, int, int, hipStream_t);
void launch_attn_fwd(const void*, const void*, const void*, const float*,
                     void*, int, int, int, int, int, int, bool, float, long,
                     long, long, long, const float*, const float*, const int*,
                     hipStream_t);
void launch_attn_varlen(const void*, const void*, const void*, void*,
                        const int*, const int*, const int*, int, int, int,
                        int, int, int, long, long, float, const float*,
                        const float*, const int*, hipStream_t);
void launch_rope(const void*, void*, const float*, const float*, const int*,
                 long, int, int, int, hipStream_t);
long score_bytes(int, int, bool);
void launch_score(const float*, void*, const float*, void*, bool, int, int, int,
                  const float**, int**, hipStream_t);
void launch_score_again(const float*, const void*, const float*, void*,
                        const int*, int, int, int, hipStream_t);
void launch_search_top(const unsigned int*, const float*, const float*, float*,
                       int*, int, int, int, int, int, const float*, int*, bool,
                       hipStream_t);
int search_few_groups(int);
void launch_search_few(const float*, const float*, float*, int*, int, int, int,
                       int, hipStream_t);
void launch_narrow_most(const float*, long, int*, hipStream_t);
void launch_narrow_rows(const float*, void*, long, int, int, int, float*,
                        hipStream_t);
long narrow_bytes(long, long, long, long);
void launch_narrow_topk(const float*, const float*, const void*, void*, float*,
                        int*, int, int, int, int, int, float, float, int,
                        hipStream_t);
int narrow_again_most();
long narrow_again_bytes(int);
void launch_narrow_again(const float*, void*, const int*, int,
                         unsigned long long*, float*, int*, int, int, int, int,
                         int, hipStream_t);
void launch_topk_chunk(const float*, const int*, float*, int*, int, long, int,
                       int, bool, hipStream_t);
void launch_hamming_score(const void*, const void*, float*, int, long, int,
                          hipStream_t);
void launch_ivf_score(const void*, const int*, const int*, const float*,
                      float*, int, int, int, int, hipStream_t);
void launch_gemv_fp8(const void*, const void*, const float*, const void*,
                     void*, int, int, long, bool, hipStream_t);
void launch_gemv_fp8_norm(const void*, const void*, const void*, void*, float,
                          const void*, const float*, const void*, void*, int,
                          int, bool, hipStream_t);
void launch_sample(const float*, const float*, int*, int, int, float, float,
                   hipStream_t);
void launch_paged_attn(const void*, long, void*, void*, const int*,
                       const int*, void*, void*, void*, int, int, int, int,
                       int, int, float, bool, bool, hipStream_t);
void launch_step_attn(const void*, const float*, int, const void*,
                      const float*, const float*, void*, void*, const int*,
                      const int*, void*, void*, void*, int*, const int*, int,
                      int, int, int, int, int, float, bool, bool, const Ahead*,
                      hipStream_t);
void launch_step_plan(const int*, const int*, int, int, int, int, int, int,
                      int*, int*, long, const void*, const void*, void*, int,
                      float, hipStream_t);
int step_plan_room(int, int, int, int);
void launch_norm_parts(const float*, int, const void*, const void*, void*,
                       void*, int, int, float, hipStream_t);
void launch_rope_put(const void*, const float*, int, const void*,
                     const float*, const float*, const int*, void*, void*,
                     void*, const int*, int, int, int, int, int, bool,
                     hipStream_t);
void launch_cache_put(const void*, const void*, void*, void*, const int*,
                      const int*, int, int, int, int, bool, hipStream_t);
}

// ---- norms ----------------------------------------------------------------
torch::Tensor norm_fwd(torch::Tensor x, c10::optional<torch::Tensor> res,
                       torch::Tensor w, c10::optional<torch::Tensor> b,
                       c10::optional<torch::Tensor> sum_out, double eps,
                       bool rms) {
  CHECK_DEV(x); CHECK_CONT(x); CHECK_BF16(x);
  const int H = x.size(-1);
  TORCH_CHECK(H % 8 == 0 && H <= 8192, "H must be mult of 8, <= 8192");
  const long n_rows = x.numel() / H;
  auto out = torch::empty_like(x);
  launch_norm_fwd(x.data_ptr(), res ? res->data_ptr() : nullptr, w.data_ptr(),
                  b ? b->data_ptr() : nullptr, out.data_ptr(),
                  sum_out ? sum_out->data_ptr() : nullptr, (int)n_rows, H,
                  (float)eps, rms, cur_stream());
  return out;
}

// slabs [S, rows, H] of a product, res [..., H] -> norm of their sum, the sum
std::vector<torch::Tensor> norm_parts(torch::Tensor parts, torch::Tensor res,
                                      torch::Tensor w, double eps) {
  CHECK_DEV(parts); CHECK_CONT(parts); CHECK_F32(parts);
  CHECK_DEV(res); CHECK_CONT(res); CHECK_BF16(res);
  CHECK_DEV(w); CHECK_CONT(w); CHECK_BF16(w);
  TORCH_CHECK(parts.dim() == 3, "parts must be [S, rows, H]");
  const int S = parts.size(0), rows = parts.size(1), H = parts.size(2);
  TORCH_CHECK(H % 8 == 0 && H <= 8192, "H must be mult of 8, <= 8192");
  TORCH_CHECK(res.numel() == (long)rows * H && res.size(-1) == H &&
                  w.numel() == H,
              "norm_parts: shape mismatch");
  auto out = torch::empty_like(res), sum = torch::empty_like(res);
  if (rows > 0)
    launch_norm_parts(parts.data_ptr<float>(), S, res.data_ptr(),
                      w.data_ptr(), out.data_ptr(), sum.data_ptr(), rows, H,
                      (float)eps, cur_stream());
  return {out, sum};
}

// ---- activations ----------------------------------------------------------
torch::Tensor bias_gelu(torch::Tensor x, c10::optional<torch::Tensor> bias,
                        bool erf) {
  CHECK_DEV(x); CHECK_CONT(x); CHECK_BF16(x);
  auto out = torch::empty_like(x);
  const int N = x.size(-1);
  TORCH_CHECK(N % 8 == 0, "last dim must be mult of 8");
  launch_bias_gelu(x.data_ptr(), bias ? bias->data_ptr() : nullptr,
                   out.data_ptr(), x.numel(), N, erf, cur_stream());
  return out;
}

torch::Tensor swiglu_packed(torch::Tensor gu) {
  CHECK_DEV(gu); CHECK_CONT(gu); CHECK_BF16(gu);
  const int I = gu.size(-1) / 2;
  TORCH_CHECK(I % 8 == 0, "I must be a multiple of 8");
  const long R = gu.numel() / (2L * I);
  auto sizes = gu.sizes().vec();
  sizes.back() = I;
  auto out = torch::empty(sizes, gu.options());
  launch_swiglu_packed(gu.data_ptr(), out.data_ptr(), R, I, cur_stream());
  return out;
}

torch::Tensor swiglu(torch::Tensor gate, torch::Tensor up) {
  CHECK_DEV(gate); CHECK_CONT(gate); CHECK_BF16(gate);
  auto out = torch::empty_like(gate);
  launch_swiglu(gate.data_ptr(), up.data_ptr(), out.data_ptr(), gate.numel(),
                cur_stream());
  return out;
}

torch::Tensor bias_add(torch::Tensor x, torch::Tensor bias) {
  CHECK_DEV(x); CHECK_CONT(x); CHECK_BF16(x);
  auto out = torch::empty_like(x);
  launch_bias_add(x.data_ptr(), bias.data_ptr(), out.data_ptr(), x.numel(),
                  x.size(-1), cur_stream());
  return out;
}

// ---- pooling ---------------------------------------------------------------
torch::Tensor mean_pool(torch::Tensor hidden, torch::Tensor mask,
                        bool normalize) {
  CHECK_DEV(hidden); CHECK_CONT(hidden); CHECK_BF16(hidden); CHECK_I32(mask);
  const int R = hidden.size(0), S = hidden.size(1), H = hidden.size(2);
  auto out = torch::empty({R, H}, hidden.options().dtype(at::kFloat));
  if (R == 0) return out;
  TORCH_CHECK(H % 8 == 0 && H <= 16384, "H must be mult of 8, <= 16384");
  TORCH_CHECK(mask.is_contiguous() && mask.numel() == (long)R * S,
              "mask must be [R, S]");
  const int NS = mean_pool_shares(R, S);
  torch::Tensor parts;
  if (NS > 1) parts = torch::empty({R, NS, H}, out.options());
  launch_mean_pool(hidden.data_ptr(), mask.data_ptr<int>(),
                   out.data_ptr<float>(),
                   NS > 1 ? parts.data_ptr<float>() : nullptr, R, S, H, NS,
                   normalize, cur_stream());
  return out;
}

torch::Tensor last_token_pool(torch::Tensor hidden, torch::Tensor mask,
                              bool left_padded, bool normalize) {
  CHECK_DEV(hidden); CHECK_CONT(hidden); CHECK_BF16(hidden); CHECK_I32(mask);
  const int R = hidden.size(0), S = hidden.size(1), H = hidden.size(2);
  auto out = torch::empty({R, H}, hidden.options().dtype(at::kFloat));
  launch_last_token_pool(hidden.data_ptr(), mask.data_ptr<int>(),
                         out.data_ptr<float>(), R, S, H, left_padded,
                         normalize, cur_stream());
  return out;
}

torch::Tensor l2_normalize(torch::Tensor x) {
  CHECK_DEV(x); CHECK_CONT(x); CHECK_F32(x);
  const int R = x.size(0), H = x.size(1);
  auto out = torch::empty_like(x);
  launch_l2_normalize(x.data_ptr<float>(), out.data_ptr<float>(), R, H,
                      cur_stream());
  return out;
}

torch::Tensor adjacent_cosine(torch::Tensor emb) {
  CHECK_DEV(emb); CHECK_CONT(emb); CHECK_F32(emb);
  const int N = emb.size(0), H = emb.size(1);
  auto out = torch::empty({std::max(N - 1, 0)},
                          emb.options().dtype(at::kFloat));
  if (N >= 2)
    launch_adjacent_cosine(emb.data_ptr<float>(), out.data_ptr<float>(), N, H,
                           cur_stream());
  return out;
}

// ---- attention -------------------------------------------------------------
static bool in_16s(const torch::Tensor& t) {
  return (uintptr_t)t.data_ptr() % 16 == 0 && t.stride(0) % 8 == 0 &&
         t.stride(1) % 8 == 0;
}

// Tables and positions by which attention rotates its queries, null if none.
struct QueryTurn {
  const float *cs = nullptr, *sn = nullptr;
  const int* pos = nullptr;
};
static QueryTurn query_turn(const c10::optional<torch::Tensor>& cs,
                            const c10::optional<torch::Tensor>& sn,
                            const c10::optional<torch::Tensor>& pos,
                            long rows, int D) {
  QueryTurn t;
  if (!cs) return t;
  TORCH_CHECK(sn && pos, "rotation: two tables and positions");
  CHECK_FLOATS((*cs)); CHECK_FLOATS((*sn)); CHECK_INTS((*pos));
  TORCH_CHECK(cs->dim() == 2 && cs->size(1) == D / 2 &&
                  cs->sizes() == sn->sizes() && pos->numel() == rows,
              "rotation tables must be [positions, D / 2], one position a row");
  t.cs = cs->data_ptr<float>();
  t.sn = sn->data_ptr<float>();
  t.pos = pos->data_ptr<int>();
  return t;
}

torch::Tensor attn_fwd(torch::Tensor Q, torch::Tensor K, torch::Tensor V,
                       c10::optional<torch::Tensor> mask, bool causal,
                       double scale, c10::optional<torch::Tensor> cs = {},
                       c10::optional<torch::Tensor> sn = {},
                       c10::optional<torch::Tensor> pos = {}) {
  // Q/K/V may be strided views (e.g. slices of a packed QKV tensor) as
  // long as the innermost (D) is contiguous and heads are D-strided.
  CHECK_DEV(Q); CHECK_BF16(Q);
  CHECK_DEV(K); CHECK_BF16(K);
  CHECK_DEV(V); CHECK_BF16(V);
  const int B = Q.size(0), SQ = Q.size(1), H = Q.size(2), D = Q.size(3);
  const int SKV = K.size(1), HKV = K.size(2);
  TORCH_CHECK(D == 64 || D == 128, "head_dim must be 64 or 128");
  TORCH_CHECK(H % HKV == 0, "GQA requires H % HKV == 0");
  TORCH_CHECK(Q.stride(3) == 1 && K.stride(3) == 1 && V.stride(3) == 1,
              "innermost dim must be contiguous");
  TORCH_CHECK(Q.stride(2) == D && K.stride(2) == D && V.stride(2) == D,
              "head stride must be D");
  TORCH_CHECK(K.stride(0) == V.stride(0) && K.stride(1) == V.stride(1),
              "K/V must share layout");
  const float* mp = nullptr;
  if (mask) {
    CHECK_DEV((*mask)); CHECK_CONT((*mask)); CHECK_F32((*mask));
    TORCH_CHECK(mask->size(0) == B && mask->size(1) == SKV,
                "mask must be [B, SKV] f32");
    mp = mask->data_ptr<float>();
  }
  auto O = torch::empty({B, SQ, H, D}, Q.options());
  // keys and values are copied 16 bytes at a time
  if (!in_16s(K) || !in_16s(V)) {
    K = K.clone(at::MemoryFormat::Contiguous);
    V = V.clone(at::MemoryFormat::Contiguous);
  }
  const QueryTurn turn = query_turn(cs, sn, pos, (long)B * SQ, D);
  launch_attn_fwd(Q.data_ptr(), K.data_ptr(), V.data_ptr(), mp, O.data_ptr(),
                  B, SQ, SKV, H, HKV, D, causal, (float)scale,
                  (long)Q.stride(0), (long)Q.stride(1), (long)K.stride(0),
                  (long)K.stride(1), turn.cs, turn.sn, turn.pos, cur_stream());
  return O;
}

torch::Tensor attn_varlen(torch::Tensor Q, torch::Tensor K, torch::Tensor V,
                          torch::Tensor cu, torch::Tensor blk_seq,
                          torch::Tensor blk_qb, double scale,
                          c10::optional<torch::Tensor> cs = {},
                          c10::optional<torch::Tensor> sn = {},
                          c10::optional<torch::Tensor> pos = {}) {
  // packed [T, H(KV), D] bf16, heads side by side in a row, rows of any
  // stride that is a multiple of 16 bytes (K's and V's the same); cu int32
  // [B+1]; blk_* int32 [nblocks]
  CHECK_DEV(Q); CHECK_BF16(Q);
  CHECK_DEV(K); CHECK_BF16(K);
  CHECK_DEV(V); CHECK_BF16(V);
  CHECK_DEV(cu); CHECK_CONT(cu);
  CHECK_DEV(blk_seq); CHECK_CONT(blk_seq);
  CHECK_DEV(blk_qb); CHECK_CONT(blk_qb);
  TORCH_CHECK(cu.scalar_type() == torch::kInt32 &&
              blk_seq.scalar_type() == torch::kInt32 &&
              blk_qb.scalar_type() == torch::kInt32,
              "cu/blk maps must be int32");
  const int T = Q.size(0), H = Q.size(1), D = Q.size(2), HKV = K.size(1);
  const int B = cu.size(0) - 1, nblocks = blk_seq.size(0);
  TORCH_CHECK(D == 64 || D == 128, "head_dim must be 64 or 128");
  TORCH_CHECK(H % HKV == 0, "GQA requires H % HKV == 0");
  for (const auto& t : {Q, K, V})
    TORCH_CHECK(t.stride(2) == 1 && t.stride(1) == D &&
                    t.stride(0) % 8 == 0 &&
                    (uintptr_t)t.data_ptr() % 16 == 0,
                "heads must be neighbours, rows aligned to 16 bytes");
  TORCH_CHECK(K.stride(0) == V.stride(0), "K/V must share layout");
  // rows past cu[B] (padding added to keep GEMM shapes 256-aligned) are not
  // covered by the block map and are zeroed
  auto O = torch::empty({T, H, D}, Q.options());
  const QueryTurn turn = query_turn(cs, sn, pos, T, D);
  launch_attn_varlen(Q.data_ptr(), K.data_ptr(), V.data_ptr(), O.data_ptr(),
                     cu.data_ptr<int>(), blk_seq.data_ptr<int>(),
                     blk_qb.data_ptr<int>(), nblocks, B, T, H, HKV, D,
                     Q.stride(0), K.stride(0), (float)scale, turn.cs, turn.sn,
                     turn.pos, cur_stream());
  return O;
}

// ---- rope ------------------------------------------------------------------
torch::Tensor rope_apply(torch::Tensor x, torch::Tensor cs, torch::Tensor sn,
                         torch::Tensor pos, int64_t rope_heads = -1) {
  CHECK_DEV(x); CHECK_CONT(x); CHECK_BF16(x);
  CHECK_F32(cs); CHECK_F32(sn); CHECK_I32(pos);
  const int D = x.size(-1);
  const int Hx = x.size(-2);
  const long n_rows = x.numel() / ((long)D * Hx) * Hx;
  auto out = torch::empty_like(x);
  launch_rope(x.data_ptr(), out.data_ptr(), cs.data_ptr<float>(),
              sn.data_ptr<float>(), pos.data_ptr<int>(), n_rows, Hx, D,
              rope_heads < 0 ? Hx : (int)rope_heads, cur_stream());
  return out;
}

// x [..., heads or more, D], rows of equal stride: the first `heads` heads of
// every row are rotated in place
void rope_inplace(torch::Tensor x, torch::Tensor cs, torch::Tensor sn,
                  torch::Tensor pos, int64_t heads, int64_t first) {
  CHECK_DEV(x); CHECK_CONT(x); CHECK_BF16(x);
  CHECK_FLOATS(cs); CHECK_FLOATS(sn); CHECK_INTS(pos);
  const int D = x.size(-1);
  const long ld = x.size(-2) * (long)D, n_rows = x.numel() / ld;
  TORCH_CHECK(D == 64 || D == 128, "head_dim must be 64 or 128");
  TORCH_CHECK(heads >= 0 && first >= 0 && first + heads <= x.size(-2) &&
                  pos.numel() == n_rows,
              "one position per row, at most its heads");
  TORCH_CHECK(cs.size(-1) == D / 2 && cs.sizes() == sn.sizes() &&
                  (uintptr_t)x.data_ptr() % 16 == 0,
              "rotation tables must be [positions, D / 2]");
  if (n_rows > 0)
    launch_rope_inplace((char*)x.data_ptr() + first * D * 2,
                        cs.data_ptr<float>(),
                        sn.data_ptr<float>(), pos.data_ptr<int>(), n_rows, ld,
                        (int)heads, D, cur_stream());
}

// ---- encoder inputs ---------------------------------------------------------
static int mask_bytes(const torch::Tensor& mask) {
  CHECK_DEV(mask); CHECK_CONT(mask);
  const int bytes = mask.element_size();
  TORCH_CHECK(!mask.is_floating_point() && !mask.is_complex() &&
                  (bytes == 1 || bytes == 4 || bytes == 8),
              "mask must be of 8, 32 or 64 bit integers or truth values");
  return bytes;
}

// The layer norm, and the key bias of a mask that is there.
static std::vector<torch::Tensor> embed_tokens(
    torch::Tensor ids, c10::optional<torch::Tensor> pos_ids,
    torch::Tensor word, torch::Tensor pos, torch::Tensor type, torch::Tensor w,
    torch::Tensor b, double eps, c10::optional<torch::Tensor> mask) {
  CHECK_DEV(ids); CHECK_CONT(ids);
  TORCH_CHECK(ids.scalar_type() == at::kLong && ids.dim() == 2,
              "ids must be int64 [B, S]");
  const int S = ids.size(1), H = word.size(1);
  for (const auto& t : {word, pos, type, w, b}) {
    CHECK_DEV(t); CHECK_CONT(t); CHECK_BF16(t);
    TORCH_CHECK(t.size(-1) == H, "equal widths");
  }
  TORCH_CHECK(H % 8 == 0 && H <= 8192, "H must be mult of 8, <= 8192");
  if (pos_ids) {
    CHECK_DEV(pos_ids.value()); CHECK_CONT(pos_ids.value());
    TORCH_CHECK(pos_ids->scalar_type() == at::kLong &&
                    pos_ids->numel() == ids.numel(),
                "pos_ids must be int64, one per token");
  } else {
    TORCH_CHECK(S <= pos.size(0), "more tokens than positions");
  }
  auto out = torch::empty({ids.size(0), S, H}, word.options());
  torch::Tensor bias;
  int bytes = 0;
  if (mask) {
    bytes = mask_bytes(*mask);
    TORCH_CHECK(mask->sizes() == ids.sizes() && mask->device() == ids.device(),
                "a mask number per token");
    bias = torch::empty(ids.sizes(), ids.options().dtype(at::kFloat));
  }
  // (rows without numbers have nothing to be asked for ahead)
  if (ids.numel() > 0 && H == 0 && mask)
    launch_key_bias(mask->data_ptr(), bias.data_ptr<float>(), mask->numel(),
                    bytes, cur_stream());
  if (ids.numel() > 0 && H > 0)
    launch_embed_layer_norm(
        (const long*)ids.data_ptr<int64_t>(),
        pos_ids ? (const long*)pos_ids->data_ptr<int64_t>() : nullptr,
        word.data_ptr(), pos.data_ptr(), type.data_ptr(), w.data_ptr(),
        b.data_ptr(), out.data_ptr(), ids.numel(), S, H, word.size(0),
        pos.size(0), (float)eps, mask ? mask->data_ptr() : nullptr, bytes,
        mask ? bias.data_ptr<float>() : nullptr, cur_stream());
  return {out, bias};
}

torch::Tensor embed_layer_norm(torch::Tensor ids,
                               c10::optional<torch::Tensor> pos_ids,
                               torch::Tensor word, torch::Tensor pos,
                               torch::Tensor type, torch::Tensor w,
                               torch::Tensor b, double eps) {
  return embed_tokens(ids, pos_ids, word, pos, type, w, b, eps,
                      c10::nullopt)[0];
}

std::vector<torch::Tensor> embed_with_bias(
    torch::Tensor ids, c10::optional<torch::Tensor> pos_ids,
    torch::Tensor word, torch::Tensor pos, torch::Tensor type, torch::Tensor w,
    torch::Tensor b, double eps, torch::Tensor mask) {
  return embed_tokens(ids, pos_ids, word, pos, type, w, b, eps, mask);
}

torch::Tensor key_bias(torch::Tensor mask) {
  const int bytes = mask_bytes(mask);
  auto out = torch::empty(mask.sizes(), mask.options().dtype(at::kFloat));
  if (mask.numel() > 0)
    launch_key_bias(mask.data_ptr(), out.data_ptr<float>(), mask.numel(),
                    bytes, cur_stream());
  return out;
}

// ---- search ----------------------------------------------------------------
// What the scores of queries [Q, K] against rows [N, K] ask.
static void check_score(const torch::Tensor& q, const torch::Tensor& corpus) {
  CHECK_DEV(q); CHECK_CONT(q); CHECK_F32(q);
  CHECK_DEV(corpus); CHECK_CONT(corpus); CHECK_F32(corpus);
  TORCH_CHECK(q.dim() == 2 && corpus.dim() == 2, "matrices");
  TORCH_CHECK(q.device() == corpus.device(), "score: two devices");
  const long Q = q.size(0), K = q.size(1), N = corpus.size(0);
  TORCH_CHECK(corpus.size(1) == K && K >= 32 && K % 32 == 0, "K % 32");
  // rows are counted in 32 bits up to the end of the last tile
  TORCH_CHECK(Q < (1L << 20) && N <= (1L << 31) - 256 && K < (1L << 20) &&
                  Q * N < (1L << 39),  // 2^24 workgroups of 256 x 128
              "score: too large");
  TORCH_CHECK((uintptr_t)q.data_ptr() % 16 == 0 &&
                  (uintptr_t)corpus.data_ptr() % 16 == 0,
              "score: 16-byte alignment");
}

torch::Tensor score(torch::Tensor q, torch::Tensor corpus) {
  check_score(q, corpus);
  // as the library's product that this stands in for
  const c10::DeviceGuard guard(q.device());
  const long Q = q.size(0), K = q.size(1), N = corpus.size(0);
  auto out = torch::empty({Q, N}, q.options());
  if (out.numel() == 0) return out;
  auto planes = torch::empty({score_bytes((int)Q, (int)K, true)},
                             q.options().dtype(at::kByte));
  const float* lost;
  int* again;
  launch_score(q.data_ptr<float>(), planes.data_ptr(),
               corpus.data_ptr<float>(), out.data_ptr(), true, (int)Q, (int)N,
               (int)K, &lost, &again, cur_stream());
  return out;
}

// The k largest scores of every query and their rows, [Q, k] each, one behind the
// other, without the scores' matrix.
std::vector<torch::Tensor> score_topk(torch::Tensor q, torch::Tensor corpus,
                                      int64_t k) {
  check_score(q, corpus);
  const c10::DeviceGuard guard(q.device());
  const long Q = q.size(0), K = q.size(1), N = corpus.size(0);
  TORCH_CHECK(Q > 0 && k > 0 && k <= 60 && k <= N, "score_topk: 1 to 60 of N");
  const long groups = (N + 127) / 128 * 32;
  const auto words = q.options().dtype(at::kInt);
  auto most = torch::empty({Q, groups}, words);
  auto both = torch::empty({2, Q, k}, words);
  auto ov = both.select(0, 0).view(at::kFloat), oi = both.select(0, 1);
  auto* at = reinterpret_cast<unsigned int*>(most.data_ptr<int>());
  auto planes = torch::empty({score_bytes((int)Q, (int)K, false)},
                             q.options().dtype(at::kByte));
  const float *qp = q.data_ptr<float>(), *cp = corpus.data_ptr<float>(), *lost;
  int* again;
  launch_score(qp, planes.data_ptr(), cp, at, false, (int)Q, (int)N, (int)K,
               &lost, &again, cur_stream());
  auto top = [&](bool second) {
    launch_search_top(at, qp, cp, ov.data_ptr<float>(), oi.data_ptr<int>(),
                      (int)Q, (int)N, (int)groups, (int)K, (int)k, lost, again,
                      second, cur_stream());
  };
  top(false);
  if (again) {
    launch_score_again(qp, planes.data_ptr(), cp, at, again, (int)Q, (int)N,
                       (int)K, cur_stream());
    top(true);
  }
  return {ov, oi};
}

// Products in float32 of up to four queries with all rows, and the k best of them.
std::vector<torch::Tensor> search_few(torch::Tensor q, torch::Tensor corpus,
                                      int64_t k) {
  for (const auto& t : {q, corpus}) {
    CHECK_DEV(t); CHECK_CONT(t); CHECK_F32(t);
    TORCH_CHECK(t.dim() == 2 && (uintptr_t)t.data_ptr() % 16 == 0 &&
                    t.device() == q.device(),
                "rows aligned to 16 bytes");
  }
  const long Q = q.size(0), K = q.size(1), N = corpus.size(0);
  TORCH_CHECK(Q > 0 && Q <= (K > 768 ? 2 : 4) && corpus.size(1) == K &&
                  K > 0 && K % 4 == 0 && K <= 1024 && N >= 64 &&
                  N < (1L << 31) - 256 && k > 0 && k <= 30,
              "search_few: sizes");
  const c10::DeviceGuard guard(q.device());
  const long of_all = search_few_groups((int)N) * (k | 1);
  const auto words = q.options().dtype(at::kInt);
  auto some = torch::empty({2, Q, of_all}, words);
  auto both = torch::empty({2, Q, k}, words);
  float* sv = reinterpret_cast<float*>(some.data_ptr<int>());
  int* si = some.data_ptr<int>() + Q * of_all;
  auto ov = both.select(0, 0).view(at::kFloat), oi = both.select(0, 1);
  launch_search_few(q.data_ptr<float>(), corpus.data_ptr<float>(), sv, si,
                    (int)Q, (int)N, (int)K, (int)k, cur_stream());
  launch_topk_chunk(sv, si, ov.data_ptr<float>(), oi.data_ptr<int>(), (int)Q,
                    of_all, 8192, (int)k, true, cur_stream());
  return {ov, oi};
}

// Rows [N, K] times the power of two that brings the largest number to 2^13, as f16
// in blocks (narrow_search.hip; [N in whole 16s, K in whole 64s] of them), that power,
// and the largest |row - row as f16| and |row as f16| (and the root of the mean square
// of the latter) of rows times it. Nothing where a number is infinite or NaN, or all
// are 0. Waits for the GPU.
c10::optional<std::tuple<torch::Tensor, int64_t, double, double, double>>
narrow_rows(torch::Tensor corpus) {
  CHECK_DEV(corpus); CHECK_CONT(corpus); CHECK_F32(corpus);
  TORCH_CHECK(corpus.dim() == 2 && corpus.size(0) > 0 && corpus.size(1) > 0 &&
                  corpus.size(1) % 4 == 0 && corpus.size(1) < (1L << 16) &&
                  (uintptr_t)corpus.data_ptr() % 16 == 0,
              "rows of fours, aligned to 16 bytes");
  const c10::DeviceGuard guard(corpus.device());
  const long N = corpus.size(0), K = corpus.size(1);
  const long KP = std::max(128L, (K + 63) / 64 * 64);
  auto facts = torch::zeros({4}, corpus.options());
  launch_narrow_most(corpus.data_ptr<float>(), N * K,
                     reinterpret_cast<int*>(facts.data_ptr<float>()) + 3,
                     cur_stream());
  const float most = facts[3].item<float>();
  if (!(most > 0.f && most <= std::numeric_limits<float>::max()))
    return c10::nullopt;
  const int up = std::min(13 - std::ilogb(most), 120);
  auto rows = torch::empty({(N + 15) / 16 * 16, KP}, corpus.options().dtype(at::kHalf));
  launch_narrow_rows(corpus.data_ptr<float>(), rows.data_ptr(), N, (int)K,
                     (int)KP, up, facts.data_ptr<float>(), cur_stream());
  const auto host = facts.cpu();
  const float* f = host.data_ptr<float>();
  return std::make_tuple(rows, (int64_t)up, std::sqrt((double)f[0]),
                         std::sqrt((double)f[1]), std::sqrt((double)f[2] / N));
}

// What narrow_topk asks (narrow_search.hip); the bytes of its workspace.
static long check_narrow(const torch::Tensor& q, const torch::Tensor& corpus,
                         const torch::Tensor& rows, int64_t up, int64_t k) {
  for (const auto& t : {corpus, rows}) {
    CHECK_DEV(t); CHECK_CONT(t);
    TORCH_CHECK(t.dim() == 2 && (uintptr_t)t.data_ptr() % 16 == 0 &&
                    t.device() == corpus.device(),
                "rows aligned to 16 bytes");
  }
  CHECK_CONT(q); CHECK_F32(q); CHECK_F32(corpus);
  TORCH_CHECK(rows.scalar_type() == at::kHalf, "rows as f16");
  const long N = corpus.size(0), K = corpus.size(1), KP = rows.size(1);
  TORCH_CHECK(q.dim() == 2 && q.size(1) == K, "queries [Q, K]");
  const long bytes = narrow_bytes(q.size(0), N, K, KP);
  TORCH_CHECK(bytes > 0 && rows.size(0) == (N + 15) / 16 * 16 && k > 0 &&
                  k <= 60 && k <= N && up >= -200 && up <= 200,
              "narrow_topk: sizes");
  return bytes;
}

// The k best rows for every query, [Q, k] scores and rows one behind the other, by
// way of the rows that narrow_rows made. A query that they cannot answer has INT_MIN
// for rows.
std::vector<torch::Tensor> narrow_topk(torch::Tensor q, torch::Tensor corpus,
                                       torch::Tensor rows, int64_t up,
                                       double error, double norm, int64_t k) {
  const long bytes = check_narrow(q, corpus, rows, up, k);
  CHECK_DEV(q);
  TORCH_CHECK((uintptr_t)q.data_ptr() % 16 == 0 &&
                  q.device() == corpus.device(),
              "queries aligned to 16 bytes");
  const c10::DeviceGuard guard(q.device());
  const long Q = q.size(0);
  auto space = torch::empty({bytes}, q.options().dtype(at::kByte));
  auto both = torch::empty({2, Q, k}, q.options().dtype(at::kInt));
  auto ov = both.select(0, 0).view(at::kFloat), oi = both.select(0, 1);
  launch_narrow_topk(q.data_ptr<float>(), corpus.data_ptr<float>(),
                     rows.data_ptr(), space.data_ptr(), ov.data_ptr<float>(),
                     oi.data_ptr<int>(), (int)Q, (int)corpus.size(0),
                     (int)q.size(1), (int)rows.size(1), (int)up, (float)error,
                     (float)norm, (int)k, cur_stream());
  return {ov, oi};
}

std::vector<torch::Tensor> topk_chunked(torch::Tensor scores,
                                        c10::optional<torch::Tensor> in_idx,
                                        int64_t k, int64_t chunk, bool regs) {
  // regs: a workgroup holds its chunk in registers; else it is read by rounds
  // of a radix select
  CHECK_DEV(scores); CHECK_CONT(scores); CHECK_F32(scores);
  TORCH_CHECK(!regs || (chunk > 0 && chunk <= 8192 && k > 0 && k <= 256),
              "chunks of up to 8192 scores and k up to 256 in registers");
  const int Q = scores.size(0);
  const long N = scores.size(1);
  const int nchunks = (int)((N + chunk - 1) / chunk);
  // one behind the other, so that one copy takes both to the host
  auto both = torch::empty({2, Q, (long)nchunks * k},
                           scores.options().dtype(at::kInt));
  auto ov = both.select(0, 0).view(at::kFloat), oi = both.select(0, 1);
  launch_topk_chunk(scores.data_ptr<float>(),
                    in_idx ? in_idx->data_ptr<int>() : nullptr,
                    ov.data_ptr<float>(), oi.data_ptr<int>(), Q, N, (int)chunk,
                    (int)k, regs, cur_stream());
  return {ov, oi};
}

torch::Tensor hamming_score(torch::Tensor qcodes, torch::Tensor codes_t) {
  CHECK_DEV(qcodes); CHECK_CONT(qcodes);
  CHECK_DEV(codes_t); CHECK_CONT(codes_t);
  TORCH_CHECK(qcodes.scalar_type() == at::kLong || qcodes.scalar_type() == at::kUInt64);
  const int Q = qcodes.size(0), W = qcodes.size(1);
  const long N = codes_t.size(1);
  auto out = torch::empty({Q, N}, qcodes.options().dtype(at::kFloat));
  launch_hamming_score(qcodes.data_ptr(), codes_t.data_ptr(),
                       out.data_ptr<float>(), Q, N, W, cur_stream());
  return out;
}

// ---- sampling / decode -----------------------------------------------------
torch::Tensor sample_tokens(torch::Tensor logits, torch::Tensor rand,
                            double temp, double min_p) {
  CHECK_DEV(logits); CHECK_CONT(logits); CHECK_F32(logits);
  const int B = logits.size(0), V = logits.size(1);
  auto out = torch::empty({B}, logits.options().dtype(at::kInt));
  launch_sample(logits.data_ptr<float>(), rand.data_ptr<float>(),
                out.data_ptr<int>(), B, V, (float)temp, (float)min_p,
                cur_stream());
  return out;
}

static void check_kv_pages(const torch::Tensor& kcache,
                           const torch::Tensor& vcache,
                           const torch::Tensor& block_table,
                           const torch::Tensor& ctx, long B, long D) {
  CHECK_DEV(kcache); CHECK_CONT(kcache);
  CHECK_DEV(vcache); CHECK_CONT(vcache);
  CHECK_SAME(kcache, vcache);
  TORCH_CHECK(kcache.scalar_type() == at::kByte ||
                  kcache.scalar_type() == at::kBFloat16,
              "pages are bf16 or fp8 (uint8)");
  TORCH_CHECK(kcache.dim() == 4 && kcache.sizes() == vcache.sizes() &&
                  kcache.size(2) == 16 && kcache.size(3) == D,
              "pages must be [blocks, HKV, 16, D]");
  CHECK_INTS(block_table);
  CHECK_INTS(ctx);
  TORCH_CHECK(block_table.dim() == 2 && block_table.size(0) == B &&
                  ctx.numel() == B,
              "one block-table row and context length per sequence");
}

// Workgroups that share a sequence in paged_attn: as many as make one for every
// CU (two where pages are fp8, whose buffers leave a CU to two), each with at
// least 256 of the positions that the block table has room for, 512 beyond eight
// of them: the table may be wide and the context short, and then every share
// costs and none gains. In us, at contexts of 64 to 200, 500, 2000 (bf16, heads
// of 128): 8 x 8 grouped heads 1 share 5.0, 9.3, 27; 4 8.3, 8.8, 19; 8 12.7, 13,
// 22. 8 x 32 heads 1 5.1, 15, 44; 2 11, 21, 46. 1 x 8 grouped heads of 2048 1 24,
// 8 10.5, 12 11.5, 16 11.1; of 8000 15 17.6, 31 19.0. 16 x 8 grouped of 100 to
// 3745 1 45, 2 31, 4 31; fp8 2 31, 4 25, 8 26. DISTLLM_PA_NSPLIT > 0 asks for a
// number (1: none; at most a page each, and 64, which is what the joining kernel
// has lanes for).
int64_t paged_attn_shares(int64_t B, int64_t H, int64_t HKV,
                          int64_t max_blocks, bool fp8) {
  const char* e = getenv("DISTLLM_PA_NSPLIT");
  const long asked = e ? atol(e) : 0;
  const long groups = std::max<long>(B * HKV * ((H / HKV + 15) / 16), 1);
  const long room =
      std::max(std::min(max_blocks / 16, (int64_t)8), max_blocks / 32);
  return std::max<long>(
      asked > 0 ? std::min<long>({asked, max_blocks, 64})
                : std::min<long>({(fp8 ? 512 : 256) / groups, room, 32}),
      1);
}

// What step_plan has to know of a decode step's attention, whose shares join in
// the launch, so that one that finds no keys costs next to nothing: the shares of
// a head group that give every CU one, of fp8 pages two (else 0), and a number
// that is asked for by DISTLLM_PA_NSPLIT (else 0). In us, shares of 4, 8, 16, 32
// (two launches, as above): 1 x 8 grouped heads, contexts of 64 6.2, 6.3, 6.3, 7.4
// (10.9); 2048 11.2, 8.3, 7.6, 8.8 (12.7); 8000 30, 18, 12.2, 10.6 (21); 8 x 8 of
// 2000 15.6, 20, 21 (22); 8 x 8 fp8 of 500 7.5, 9.5, 17 (11), of 2000 12.4, 12.1,
// 18.5 (18).
struct StepShares {
  int narrow, wide, asked, room;
};
static StepShares step_shares(int64_t B, int64_t H, int64_t HKV,
                              int64_t max_blocks, bool fp8) {
  const char* e = getenv("DISTLLM_PA_NSPLIT");
  const long groups = std::max<long>(HKV * ((H / HKV + 15) / 16), 1);
  StepShares s;
  s.narrow = (int)std::max<long>(256 / groups, 1);
  s.wide = fp8 ? (int)std::max<long>(512 / groups, 1) : 0;
  s.asked = e && atol(e) > 0
                ? (int)std::min<long>({atol(e), std::max<long>(max_blocks, 1), 64})
                : 0;
  s.room = step_plan_room((int)B, s.narrow, s.wide, s.asked);
  return s;
}

// What the attention launches of a decode step of `layers` layers need:
// [room, 8] shares and what PaStep says of them, and zeros [layers, B * HKV * groups of 16 query heads], a row
// of which each launch uses up.
// With x [B, 1, n], also its RMS norm times w.
std::vector<torch::Tensor> step_plan(torch::Tensor ctx,
                                     torch::Tensor block_table, int64_t layers,
                                     int64_t H, int64_t HKV, bool fp8,
                                     c10::optional<torch::Tensor> x,
                                     c10::optional<torch::Tensor> w,
                                     double eps) {
  CHECK_INTS(ctx);
  CHECK_INTS(block_table);
  TORCH_CHECK(HKV > 0 && H % HKV == 0, "GQA requires H % HKV == 0");
  const int64_t B = ctx.numel();
  TORCH_CHECK(block_table.dim() == 2 && block_table.size(0) == B &&
                  block_table.device() == ctx.device(),
              "block_table must be [B, blocks]");
  const int64_t max_blocks = block_table.size(1);
  const StepShares s = step_shares(B, H, HKV, max_blocks, fp8);
  auto slots = torch::empty({s.room, 8}, ctx.options());
  auto arrived = torch::empty({layers, B * HKV * ((H / HKV + 15) / 16)},
                              ctx.options());
  std::vector<torch::Tensor> out = {slots, arrived};
  torch::Tensor h;
  if (x) {
    TORCH_CHECK(w, "rows come with the norm's weights");
    for (const auto& t : {*x, *w}) {
      CHECK_DEV(t); CHECK_CONT(t); CHECK_BF16(t);
      TORCH_CHECK((uintptr_t)t.data_ptr() % 16 == 0 &&
                      t.device() == ctx.device(),
                  "16-byte alignment");
    }
    TORCH_CHECK(x->dim() == 3 && x->size(0) == B && x->size(1) == 1 &&
                    x->size(2) == w->numel() && w->numel() > 0 &&
                    w->numel() % 8 == 0 && w->numel() <= 8192,
                "rows must be [B, 1, n], n % 8 == 0 and up to 8192");
    h = torch::empty_like(*x);
    out.push_back(h);
  }
  if (B > 0)
    launch_step_plan(
        ctx.data_ptr<int>(), block_table.data_ptr<int>(), (int)B,
        (int)max_blocks, s.room, s.narrow, s.wide, s.asked,
        slots.data_ptr<int>(), arrived.data_ptr<int>(), arrived.numel(),
        x ? x->data_ptr() : nullptr, x ? w->data_ptr() : nullptr,
        x ? h.data_ptr() : nullptr, x ? (int)w->numel() : 0, (float)eps,
        cur_stream());
  return out;
}

torch::Tensor paged_attn(torch::Tensor q, torch::Tensor kcache,
                         torch::Tensor vcache, torch::Tensor block_table,
                         torch::Tensor ctx_len, double scale) {
  CHECK_DEV(q); CHECK_CONT(q); CHECK_BF16(q);
  const int B = q.size(0), H = q.size(1), D = q.size(2);
  const int HKV = kcache.size(1);
  const int max_blocks = block_table.size(1);
  TORCH_CHECK(D == 64 || D == 128, "head_dim must be 64 or 128");
  TORCH_CHECK(H % HKV == 0, "GQA requires H % HKV == 0");
  check_kv_pages(kcache, vcache, block_table, ctx_len, B, D);
  const bool fp8 = kcache.scalar_type() == at::kByte;
  auto out = torch::empty_like(q);
  if (B == 0) return out;
  q = aligned16(q);
  const bool aligned = (uintptr_t)kcache.data_ptr() % 16 == 0 &&
                       (uintptr_t)vcache.data_ptr() % 16 == 0;
  const int NS = (int)paged_attn_shares(B, H, HKV, max_blocks, fp8);
  torch::Tensor pacc, pml;
  if (NS > 1) {
    auto f32 = q.options().dtype(at::kFloat);
    pacc = torch::empty({(long)B * H * NS, D}, f32);
    pml = torch::empty({(long)B * H * NS, 2}, f32);
  }
  launch_paged_attn(q.data_ptr(), q.stride(0), kcache.data_ptr(),
                    vcache.data_ptr(), block_table.data_ptr<int>(),
                    ctx_len.data_ptr<int>(), out.data_ptr(),
                    NS > 1 ? pacc.data_ptr() : nullptr,
                    NS > 1 ? pml.data_ptr() : nullptr, B, H, HKV, D,
                    max_blocks, NS, (float)scale, fp8, aligned, cur_stream());
  return out;
}

// qkv [B, H + 2 HKV, D] of a decode step, or the slabs [S, B, H + 2 HKV, D]
// fp32 of the product that it would be, and its bias
struct StepSizes {
  bool parts;
  int B, H, HKV, D;
};
static StepSizes check_step(const torch::Tensor& qkv, const torch::Tensor& cs,
                            const torch::Tensor& sn, const torch::Tensor& ctx,
                            const torch::Tensor& kcache,
                            const torch::Tensor& vcache,
                            const torch::Tensor& block_table,
                            const c10::optional<torch::Tensor>& bias) {
  CHECK_DEV(qkv); CHECK_CONT(qkv);
  CHECK_FLOATS(cs); CHECK_FLOATS(sn);
  const bool parts = qkv.scalar_type() == at::kFloat;
  if (!parts) CHECK_BF16(qkv);
  TORCH_CHECK(qkv.dim() == 3 + parts, "qkv must be [B, H + 2 HKV, D]");
  TORCH_CHECK(!bias || parts, "a bias goes with slabs");
  const int B = qkv.size(parts), D = qkv.size(2 + parts);
  const int HKV = kcache.size(1), H = (int)qkv.size(1 + parts) - 2 * HKV;
  TORCH_CHECK(D == 64 || D == 128, "head_dim must be 64 or 128");
  TORCH_CHECK(H > 0, "qkv must be [B, H + 2 HKV, D]");
  TORCH_CHECK(cs.size(-1) == D / 2 && cs.sizes() == sn.sizes(),
              "rotation tables must be [positions, D / 2]");
  check_kv_pages(kcache, vcache, block_table, ctx, B, D);
  if (bias) {
    CHECK_DEV(bias.value()); CHECK_CONT(bias.value());
    CHECK_BF16(bias.value());
    TORCH_CHECK(bias->numel() == (long)(H + 2 * HKV) * D, "bias");
  }
  return {parts, B, H, HKV, D};
}

// -> rotated q [B, H, D]; rotated keys and the values to their places (position
// ctx - 1) in the cache
torch::Tensor rope_put(torch::Tensor qkv, torch::Tensor cs, torch::Tensor sn,
                       torch::Tensor ctx, torch::Tensor kcache,
                       torch::Tensor vcache, torch::Tensor block_table,
                       c10::optional<torch::Tensor> bias) {
  const StepSizes z =
      check_step(qkv, cs, sn, ctx, kcache, vcache, block_table, bias);
  auto q = torch::empty({z.B, z.H, z.D}, qkv.options().dtype(at::kBFloat16));
  if (z.B > 0)
    launch_rope_put(z.parts ? nullptr : qkv.data_ptr(),
                    z.parts ? qkv.data_ptr<float>() : nullptr,
                    z.parts ? (int)qkv.size(0) : 0,
                    bias ? bias->data_ptr() : nullptr, cs.data_ptr<float>(),
                    sn.data_ptr<float>(), ctx.data_ptr<int>(), q.data_ptr(),
                    kcache.data_ptr(), vcache.data_ptr(),
                    block_table.data_ptr<int>(), z.B, z.H, z.HKV, z.D,
                    block_table.size(1), kcache.scalar_type() == at::kByte,
                    cur_stream());
  return q;
}

// Weights [N, K] that a product of few rows reads next, as runs of the 16 rows that
// its workgroups have; nothing where they cannot be read in pieces of 1 KiB. Of
// large ones the first 40 MiB, what an attention of 8 us leaves the time for.
static Ahead ahead_of(const c10::optional<torch::Tensor>& w,
                      const torch::Tensor& like) {
  if (!w || w->dim() != 2 || !w->is_contiguous() ||
      w->device() != like.device() || (uintptr_t)w->data_ptr() % 16)
    return Ahead{};
  const long run = 16 * w->size(1) * w->element_size();
  if (run == 0 || run % 1024) return Ahead{};
  const long chunks = std::min<long>(w->size(0) / 16, (40l << 20) / run);
  if (chunks < 8) return Ahead{};
  return Ahead{(const char*)w->data_ptr(), 192, (int)chunks,
               (int)(run / 1024)};
}

// rope_put and the attention of its queries [B, H, D] in one launch. slots and
// arrived: of step_plan for the same lengths, heads and block table. ahead: the
// weights [N, K] of the product that follows, for the caches.
torch::Tensor step_attn(torch::Tensor qkv, torch::Tensor cs, torch::Tensor sn,
                        torch::Tensor ctx, torch::Tensor kcache,
                        torch::Tensor vcache, torch::Tensor block_table,
                        c10::optional<torch::Tensor> bias, double scale,
                        torch::Tensor slots, torch::Tensor arrived,
                        c10::optional<torch::Tensor> ahead) {
  const StepSizes z =
      check_step(qkv, cs, sn, ctx, kcache, vcache, block_table, bias);
  TORCH_CHECK(z.H % z.HKV == 0, "GQA requires H % HKV == 0");
  const int max_blocks = block_table.size(1);
  const bool fp8 = kcache.scalar_type() == at::kByte;
  auto out =
      torch::empty({z.B, z.H, z.D}, qkv.options().dtype(at::kBFloat16));
  if (z.B == 0) return out;
  CHECK_INTS(slots);
  CHECK_INTS(arrived);
  const int room = slots.size(0);
  TORCH_CHECK(slots.dim() == 2 && slots.size(1) == 8 && room >= z.B &&
                  (uintptr_t)slots.data_ptr() % 16 == 0,
              "slots: those of step_plan");
  TORCH_CHECK(arrived.numel() >= (long)z.B * z.HKV * ((z.H / z.HKV + 15) / 16),
              "arrived: one for every group of heads");
  auto f32 = qkv.options().dtype(at::kFloat);
  auto pacc = torch::empty({(long)room * z.H, z.D}, f32);
  auto pml = torch::empty({(long)room * z.H, 2}, f32);
  qkv = aligned16(qkv);
  cs = aligned16(cs);
  sn = aligned16(sn);
  const bool aligned = (uintptr_t)kcache.data_ptr() % 16 == 0 &&
                       (uintptr_t)vcache.data_ptr() % 16 == 0;
  const Ahead next = z.B <= 8 ? ahead_of(ahead, qkv) : Ahead{};
  launch_step_attn(z.parts ? nullptr : qkv.data_ptr(),
                   z.parts ? qkv.data_ptr<float>() : nullptr,
                   z.parts ? (int)qkv.size(0) : 0,
                   bias ? bias->data_ptr() : nullptr, cs.data_ptr<float>(),
                   sn.data_ptr<float>(), kcache.data_ptr(), vcache.data_ptr(),
                   block_table.data_ptr<int>(), ctx.data_ptr<int>(),
                   out.data_ptr(), pacc.data_ptr(), pml.data_ptr(),
                   arrived.data_ptr<int>(), slots.data_ptr<int>(), room, z.B,
                   z.H, z.HKV, z.D, max_blocks, (float)scale, fp8, aligned,
                   &next, cur_stream());
  return out;
}

void cache_put(torch::Tensor knew, torch::Tensor vnew, torch::Tensor kcache,
               torch::Tensor vcache, torch::Tensor block_table,
               torch::Tensor slot) {
  CHECK_DEV(knew); CHECK_CONT(knew); CHECK_BF16(knew);
  const int B = knew.size(0), HKV = knew.size(1), D = knew.size(2);
  const bool fp8 = kcache.scalar_type() == at::kByte;
  launch_cache_put(knew.data_ptr(), vnew.data_ptr(), kcache.data_ptr(),
                   vcache.data_ptr(), block_table.data_ptr<int>(),
                   slot.data_ptr<int>(), B, HKV, D, block_table.size(1),
                   fp8, cur_stream());
}

torch::Tensor ivf_score(torch::Tensor slabs, torch::Tensor lens,
                        torch::Tensor probes, torch::Tensor q) {
  CHECK_DEV(slabs); CHECK_CONT(slabs); CHECK_F32(slabs);
  CHECK_DEV(lens); CHECK_CONT(lens); CHECK_I32(lens);
  CHECK_DEV(probes); CHECK_CONT(probes); CHECK_I32(probes);
  CHECK_DEV(q); CHECK_CONT(q); CHECK_F32(q);
  const int cap = slabs.size(1), H = slabs.size(2);
  const int Q = probes.size(0), nprobe = probes.size(1);
  TORCH_CHECK(H % 4 == 0, "slab dim must be padded to a multiple of 4");
  TORCH_CHECK(q.size(0) == Q && q.size(1) == H, "q shape mismatch");
  auto out = torch::empty({Q, nprobe, cap},
                          q.options().dtype(at::kFloat));
  launch_ivf_score(slabs.data_ptr(), lens.data_ptr<int>(),
                   probes.data_ptr<int>(), q.data_ptr<float>(),
                   out.data_ptr<float>(), Q * nprobe, nprobe, cap, H,
                   cur_stream());
  return out;
}

torch::Tensor gemv_fp8(torch::Tensor x, torch::Tensor wq,
                       torch::Tensor scale,
                       c10::optional<torch::Tensor> bias, bool swiglu) {
  CHECK_DEV(x); CHECK_CONT(x); CHECK_BF16(x);
  CHECK_DEV(wq); CHECK_CONT(wq);
  TORCH_CHECK(wq.scalar_type() == at::kByte, "wq must be uint8 (fp8)");
  CHECK_DEV(scale); CHECK_CONT(scale); CHECK_F32(scale);
  const int M = x.size(0), N = wq.size(0);
  const long K = wq.size(1);
  TORCH_CHECK(x.size(1) == K, "K mismatch");
  TORCH_CHECK(M >= 1 && M <= 8, "gemv_fp8 serves M <= 8 decode rows");
  TORCH_CHECK(K % 16 == 0, "K must be a multiple of 16");
  TORCH_CHECK(scale.size(0) == N, "scale must be per output channel");
  const void* bptr = nullptr;
  if (bias.has_value()) {
    CHECK_DEV(bias.value()); CHECK_CONT(bias.value());
    CHECK_BF16(bias.value());
    TORCH_CHECK(bias->size(0) == N, "bias shape");
    bptr = bias->data_ptr();
  }
  TORCH_CHECK(!swiglu || (N % 2 == 0 && K % 128 == 0),
              "swiglu needs two halves and K % 128 == 0");
  auto out = torch::empty({M, swiglu ? N / 2 : N}, x.options());
  x = aligned16(x);
  wq = aligned16(wq);
  launch_gemv_fp8(x.data_ptr(), wq.data_ptr(),
                  scale.data_ptr<float>(), bptr, out.data_ptr(), M, N,
                  K, swiglu, cur_stream());
  return out;
}

// x = a + b, one row, and the quantized product of its RMS norm
std::vector<torch::Tensor> gemv_fp8_norm(torch::Tensor a, torch::Tensor b,
                                         torch::Tensor w_norm, double eps,
                                         torch::Tensor wq,
                                         torch::Tensor scale,
                                         c10::optional<torch::Tensor> bias,
                                         bool swiglu) {
  for (const auto& t : {a, b, w_norm}) {
    CHECK_DEV(t); CHECK_CONT(t); CHECK_BF16(t);
    TORCH_CHECK((uintptr_t)t.data_ptr() % 16 == 0, "16-byte alignment");
  }
  CHECK_DEV(wq); CHECK_CONT(wq);
  TORCH_CHECK(wq.scalar_type() == at::kByte && wq.dim() == 2 &&
                  (uintptr_t)wq.data_ptr() % 16 == 0,
              "wq must be uint8 (fp8)");
  CHECK_DEV(scale); CHECK_CONT(scale); CHECK_F32(scale);
  const int N = wq.size(0), K = wq.size(1);
  TORCH_CHECK(K % 128 == 0 && K >= 2560 && K <= 8192 && a.numel() == K &&
                  b.numel() == K && w_norm.numel() == K,
              "gemv_fp8_norm: one row of 2560 to 8192 numbers");
  TORCH_CHECK(scale.numel() == N && N > 0 && (!swiglu || N % 2 == 0),
              "scale must be per output channel");
  if (bias) {
    CHECK_DEV(bias.value()); CHECK_CONT(bias.value());
    CHECK_BF16(bias.value());
    TORCH_CHECK(bias->numel() == N, "bias");
  }
  auto out = torch::empty({1, swiglu ? N / 2 : N}, a.options());
  auto sum = torch::empty_like(b);
  launch_gemv_fp8_norm(a.data_ptr(), b.data_ptr(), w_norm.data_ptr(),
                       sum.data_ptr(), (float)eps, wq.data_ptr(),
                       scale.data_ptr<float>(),
                       bias ? bias->data_ptr() : nullptr, out.data_ptr(), N,
                       K, swiglu, cur_stream());
  return {out, sum};
}

// encoder_layers.cpp
c10::optional<torch::Tensor> bert_few_rows(torch::Tensor x,
                                           torch::Tensor mask,
                                           std::vector<torch::Tensor> layers,
                                           int64_t heads, double eps,
                                           int64_t act);

// Lists of the rows of [Q, k] scores and indices, without the entries whose index is
// negative.
static std::pair<py::list, py::list> lists_of(const float* scores,
                                              const int* indices, int64_t Q,
                                              int64_t k) {
  py::list all_scores(Q), all_indices(Q);
  for (int64_t q = 0; q < Q; ++q, scores += k, indices += k) {
    const int64_t kept =
        k - std::count_if(indices, indices + k, [](int x) { return x < 0; });
    py::list s(kept), x(kept);
    for (int64_t j = 0, to = 0; j < k; ++j) {
      if (indices[j] < 0) continue;
      PyList_SET_ITEM(s.ptr(), to, py::float_(scores[j]).release().ptr());
      PyList_SET_ITEM(x.ptr(), to++, py::int_(indices[j]).release().ptr());
    }
    all_scores[q] = std::move(s);
    all_indices[q] = std::move(x);
  }
  return {all_scores, all_indices};
}

// Scores and indices [Q, k] of a search as lists of their rows, without the
// entries whose index is negative. One copy to the host (25 us whatever it holds)
// of both, joined on the way if they do not lie one behind the other. As steps of
// Python this took a first call on a new question, which finds the host's caches
// full of other things, 60 us longer than two copies.
static std::pair<py::list, py::list> found_lists(torch::Tensor v,
                                                 torch::Tensor i) {
  CHECK_DEV(v); CHECK_F32(v);
  CHECK_DEV(i); CHECK_I32(i);
  TORCH_CHECK(v.dim() == 2 && v.sizes() == i.sizes() &&
                  v.device() == i.device(),
              "scores and indices must be [Q, k]");
  const int64_t Q = v.size(0), k = v.size(1), n = Q * k;
  torch::Tensor host;
  {
    py::gil_scoped_release others;
    const c10::DeviceGuard guard(v.device());
    const bool lie = v.is_contiguous() && i.is_contiguous() &&
                     i.is_alias_of(v) &&
                     i.storage_offset() == v.storage_offset() + n;
    host = (lie ? torch::as_strided(i, {2, Q, k}, {n, k, 1},
                                    v.storage_offset())
                : torch::stack({v.contiguous().view(at::kInt), i}))
               .cpu();
  }
  const int* at = host.data_ptr<int>();
  return lists_of(reinterpret_cast<const float*>(at), at + n, Q, k);
}

// Pinned memory of torch's cache; none where the host or a limit on locked memory does
// not give it, and nothing is left of that failure.
static c10::optional<torch::Tensor> pinned(std::vector<int64_t> size,
                                           at::ScalarType type) {
  try {
    return torch::empty(
        size, torch::TensorOptions().dtype(type).pinned_memory(true));
  } catch (const c10::Error&) {
    (void)hipGetLastError();
    return c10::nullopt;
  }
}

// found_lists of narrow_topk of queries that the host has, in one call: the GPU reads
// them and writes its answer where the host has them (pinned memory of torch's cache,
// given back when the stream has been waited for), which spares two copies and their
// waits. Above 16 MB they are copied (pinned memory stays with the process), and where
// there is none. us of 250000 rows of 768, the same work by way of copies and
// found_lists, and so: one query 111 and 96, 256 228 and 204 (score_topk 173 and 455).
// With rest: queries that narrow_topk left for near rows are asked again, one that is
// all 0 has the first rows with scores of 0, and those that are still unanswered are
// returned, as a third list, with nothing in their lists. Without, nothing (None) if
// narrow_topk left one.
static py::object narrow_found(torch::Tensor q, torch::Tensor corpus,
                               torch::Tensor rows, int64_t up, double error,
                               double norm, int64_t k, bool rest) {
  const long bytes = check_narrow(q, corpus, rows, up, k);
  TORCH_CHECK(q.device().is_cpu(), "queries of the host");
  const int64_t Q = q.size(0), K = q.size(1), n = Q * k;
  torch::Tensor answer;
  std::vector<int> left;
  {
    py::gil_scoped_release others;
    const c10::DeviceGuard guard(corpus.device());
    c10::optional<torch::Tensor> host[2];
    if (std::max(Q * K, 2 * n) <= 1 << 22) {
      host[0] = pinned({Q, K}, at::kFloat);
      if (host[0]) host[1] = pinned({2, Q, k}, at::kInt);
    }
    const bool pin = host[1].has_value();
    auto place = [&](int i, at::IntArrayRef size, at::ScalarType t) {
      return pin ? *host[i] : torch::empty(size, corpus.options().dtype(t));
    };
    auto asked = place(0, {Q, K}, at::kFloat);
    auto told = place(1, {2, Q, k}, at::kInt);
    if (pin)
      std::memcpy(asked.data_ptr(), q.data_ptr(), Q * K * sizeof(float));
    else
      asked.copy_(q);
    auto seen = [&](const torch::Tensor& t) {
      void* p = t.data_ptr();
      if (pin) C10_HIP_CHECK(hipHostGetDevicePointer(&p, t.data_ptr(), 0));
      return p;
    };
    auto space = torch::empty({bytes}, corpus.options().dtype(at::kByte));
    int* to = (int*)seen(told);
    const hipStream_t stream = cur_stream();
    const int N = (int)corpus.size(0), KP = (int)rows.size(1);
    launch_narrow_topk((const float*)seen(asked), corpus.data_ptr<float>(),
                       rows.data_ptr(), space.data_ptr(), (float*)to, to + n,
                       (int)Q, N, (int)K, KP, (int)up, (float)error,
                       (float)norm, (int)k, stream);
    // (waited for also where a launch failed: the others read what is given back)
    auto wait = [&]() {
      const hipError_t launched = hipGetLastError();
      C10_HIP_CHECK(hipStreamSynchronize(stream));
      C10_HIP_CHECK(launched);
      answer = pin ? told : told.cpu();
    };
    // of those in question the ones whose last row is not known
    auto unanswered = [&](const std::vector<int>* asked) {
      std::vector<int> out;
      const int* last = answer.data_ptr<int>() + n + k - 1;
      for (int64_t i = 0; i < (asked ? (int64_t)asked->size() : Q); ++i) {
        const int query = asked ? (*asked)[i] : (int)i;
        if (last[query * k] == INT_MIN) out.push_back(query);
      }
      return out;
    };
    wait();
    left = unanswered(nullptr);
    if (rest && !left.empty()) {
      const auto zeros = std::stable_partition(
          left.begin(), left.end(), [&](int i) {
            const float* x = q.data_ptr<float>() + i * K;
            return !std::all_of(x, x + K, [](float f) { return f == 0.f; });
          });
      const std::vector<int> first(zeros, left.end());
      left.erase(zeros, left.end());
      // (behind these, those that are left for their numbers)
      const auto other = std::stable_partition(
          left.begin(), left.end(), [&](int i) {
            return answer.data_ptr<int>()[i * k] != 0x7f800000;
          });
      const int many = (int)(other - left.begin());
      if (many > 0 && many <= narrow_again_most()) {
        auto lists = torch::empty({many * narrow_again_bytes((int)k)},
                                  space.options());
        launch_narrow_again(corpus.data_ptr<float>(), space.data_ptr(),
                            left.data(), many,
                            (unsigned long long*)lists.data_ptr(), (float*)to,
                            to + n, (int)Q, N, (int)K, KP, (int)k, stream);
        wait();
        left = unanswered(&left);
      }
      std::sort(left.begin(), left.end());
      int* found = answer.data_ptr<int>() + n;
      for (const int i : first) {
        std::iota(found + i * k, found + (i + 1) * k, 0);
        std::fill_n(found - n + i * k, k, 0);  // (the bits of 0.f)
      }
      for (const int i : left) std::fill_n(found + i * k, k, INT_MIN);
    }
  }
  if (!rest && !left.empty()) return py::none();
  const int* at = answer.data_ptr<int>();
  const auto lists = lists_of(reinterpret_cast<const float*>(at), at + n, Q, k);
  if (!rest) return py::make_tuple(lists.first, lists.second);
  return py::make_tuple(lists.first, lists.second, py::cast(left));
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("norm_fwd", &norm_fwd, "fused residual+LayerNorm/RMSNorm");
  m.def("bias_gelu", &bias_gelu);
  m.def("swiglu", &swiglu);
  m.def("swiglu_packed", &swiglu_packed);
  m.def("bias_add", &bias_add);
  m.def("mean_pool", &mean_pool);
  m.def("last_token_pool", &last_token_pool);
  m.def("l2_normalize", &l2_normalize);
  m.def("adjacent_cosine", &adjacent_cosine);
  m.def("attn_fwd", &attn_fwd, py::arg("Q"), py::arg("K"), py::arg("V"),
        py::arg("mask"), py::arg("causal"), py::arg("scale"),
        py::arg("cs") = py::none(),
        py::arg("sn") = py::none(), py::arg("pos") = py::none());
  m.def("attn_varlen", &attn_varlen, py::arg("Q"), py::arg("K"),
        py::arg("V"), py::arg("cu"), py::arg("blk_seq"), py::arg("blk_qb"),
        py::arg("scale"), py::arg("cs") = py::none(),
        py::arg("sn") = py::none(), py::arg("pos") = py::none());
  m.def("rope_apply", &rope_apply, py::arg("x"), py::arg("cs"),
        py::arg("sn"), py::arg("pos"), py::arg("rope_heads") = -1);
  m.def("rope_inplace", &rope_inplace, py::arg("x"), py::arg("cs"),
        py::arg("sn"), py::arg("pos"), py::arg("heads"), py::arg("first") = 0);
  m.def("embed_layer_norm", &embed_layer_norm, py::arg("ids"),
        py::arg("pos_ids"), py::arg("word"), py::arg("pos"), py::arg("type"),
        py::arg("w"), py::arg("b"), py::arg("eps"));
  m.def("embed_with_bias", &embed_with_bias);
  m.def("key_bias", &key_bias);
  m.def("bert_few_rows", &bert_few_rows);
  m.def("score", &score);
  m.def("score_topk", &score_topk);
  m.def("search_few", &search_few);
  m.def("narrow_rows", &narrow_rows);
  m.def("narrow_topk", &narrow_topk);
  m.def("narrow_bytes", &narrow_bytes);
  m.def("topk_chunked", &topk_chunked, py::arg("scores"), py::arg("in_idx"),
        py::arg("k"), py::arg("chunk"), py::arg("regs") = false);
  m.def("hamming_score", &hamming_score);
  m.def("ivf_score", &ivf_score);
  m.def("gemv_fp8", &gemv_fp8, py::arg("x"), py::arg("wq"),
        py::arg("scale"), py::arg("bias") = py::none(),
        py::arg("swiglu") = false);
  m.def("gemv_fp8_norm", &gemv_fp8_norm);
  m.def("sample_tokens", &sample_tokens);
  m.def("paged_attn", &paged_attn);
  m.def("paged_attn_shares", &paged_attn_shares);
  m.def("cache_put", &cache_put);
  m.def("norm_parts", &norm_parts);
  m.def("step_attn", &step_attn, py::arg("qkv"), py::arg("cs"), py::arg("sn"),
        py::arg("ctx"), py::arg("kcache"), py::arg("vcache"),
        py::arg("block_table"), py::arg("bias"), py::arg("scale"),
        py::arg("slots"), py::arg("arrived"), py::arg("ahead") = py::none());
  m.def("step_plan", &step_plan, py::arg("ctx"), py::arg("block_table"),
        py::arg("layers"), py::arg("H"), py::arg("HKV"), py::arg("fp8"),
        py::arg("x") = py::none(), py::arg("w") = py::none(),
        py::arg("eps") = 0.0);
  m.def("found_lists", &found_lists);
  m.def("pinned", [](int64_t n) { return pinned({n}, at::kByte); });
  m.def("narrow_found", &narrow_found, py::arg("q"), py::arg("corpus"),
        py::arg("rows"), py::arg("up"), py::arg("error"), py::arg("norm"),
        py::arg("k"), py::arg("rest") = false);
  m.def("rope_put", &rope_put, py::arg("qkv"), py::arg("cs"), py::arg("sn"),
        py::arg("ctx"), py::arg("kcache"), py::arg("vcache"),
        py::arg("block_table"), py::arg("bias") = py::none());
}
