// All layers of a BERT-class encoder on few rows (a question: one text, a few
// dozen tokens) in one call. Seven launches a layer of 2 to 5 us each were
// issued one by one from Python at 8 us apiece, so the GPU waited for the
// host: 1 x 24 tokens through 12 layers of 768 took 750 us, of which it
// computed 300. Here they follow each other at the cost of a launch, on
// buffers that live as long as the call, and norms and the attention of short
// texts go with the product behind them (encoder_rows.hip): 387 to 318 us, and
// 289 as what these launches wait for, and the columns of a workgroup, became less.
#include "ext_common.h"
#include "gelu_rows.h"

extern "C" {
void launch_norm_fwd(const void*, const void*, const void*, const void*,
                     void*, void*, int, int, float, bool, hipStream_t);
void launch_attn_fwd(const void*, const void*, const void*, const float*,
                     void*, int, int, int, int, int, int, bool, float, long,
                     long, long, long, const float*, const float*, const int*,
                     hipStream_t);
void launch_decode_gemm(const void*, const void*, const void*, void*, void*,
                        int, int, int, int, int, int, float, float, float,
                        const float*, const RowsArgs*, hipStream_t);
int decode_gemm_shares(int, int, int);
bool decode_gemm_rings(int, int, int);
bool norm_rows_fit(int, int);
bool attn_rows_fit(int, int, int, int);
void launch_norm_rows(const void*, const void*, const void*, const void*,
                      void*, float, const void*, const void*, void*, int, int,
                      int, int, hipStream_t);
void launch_attn_rows(const void*, const float*, const void*, const void*,
                      void*, int, int, int, int, float, hipStream_t);
}

// x [B, S, H]; mask [B, S] additive; layers: wqkv, bqkv, wo, bo, ln1_w, ln1_b,
// w1, b1, w2, b2, ln2_w, ln2_b of every layer in turn; act: decode_gemm's code
// of the feed-forward's activation. Nothing where a layer's tensors are not
// contiguous bf16 ones of the first layer's sizes: layers one by one take those.
c10::optional<torch::Tensor> bert_few_rows(torch::Tensor x,
                                           torch::Tensor mask,
                                           std::vector<torch::Tensor> layers,
                                           int64_t heads, double eps,
                                           int64_t act) {
  CHECK_DEV(x); CHECK_CONT(x); CHECK_BF16(x);
  CHECK_FLOATS(mask);
  TORCH_CHECK(x.dim() == 3, "x must be [B, S, H]");
  const int B = x.size(0), S = x.size(1), H = x.size(2), M = B * S;
  const int D = H / (int)heads;
  TORCH_CHECK(H % heads == 0 && (D == 64 || D == 128), "head size");
  TORCH_CHECK(mask.numel() == M && mask.size(0) == B, "mask must be [B, S]");
  TORCH_CHECK(M >= 1 && M <= 64 && H % 64 == 0 && H <= 8192, "x size");
  TORCH_CHECK(layers.size() % 12 == 0 && !layers.empty(),
              "twelve tensors per layer");
  TORCH_CHECK(act == 6 || act == 7, "activation");
  TORCH_CHECK(layers[6].dim() == 2 && layers[6].size(0) % 64 == 0,
              "feed-forward size");
  const long I = layers[6].size(0);
  const long rows[12] = {3L * H, 3L * H, H, H, H, H, I, I, H, H, H, H};
  const long cols[12] = {H, 0, H, 0, 0, 0, H, 0, I, 0, 0, 0};
  for (size_t i = 0; i < layers.size(); ++i) {
    const auto& t = layers[i];
    const int k = i % 12;
    if (!(t.device() == x.device() && t.scalar_type() == at::kBFloat16 &&
          t.is_contiguous() && t.dim() == (cols[k] ? 2 : 1) &&
          t.size(0) == rows[k] && (cols[k] == 0 || t.size(1) == cols[k])))
      return c10::nullopt;
    layers[i] = aligned16(t);
  }
  auto some = [&](long n) { return torch::empty({M, n}, x.options()); };
  auto qkv = some(3 * H), ctx = some(H), y = some(H), a = some(H),
       h = some(I), z = torch::empty_like(x);
  auto shares = [&](int n, int k) { return decode_gemm_shares(M, n, k); };
  const long slab = std::max(
      std::max((long)shares(3 * H, H) * 3 * H, (long)shares(H, H) * H),
      std::max((long)shares(I, H) * I, (long)shares(H, I) * H));
  auto slabs = torch::empty({slab, (long)M}, x.options().dtype(at::kFloat));
  const hipStream_t st = cur_stream();
  auto gemm = [&](const torch::Tensor& in, const torch::Tensor& w,
                  const torch::Tensor& b, torch::Tensor& out, int code) {
    const int n = w.size(0), k = w.size(1);
    launch_decode_gemm(in.data_ptr(), w.data_ptr(), b.data_ptr(),
                       out.data_ptr(), slabs.data_ptr(), M, n, k,
                       shares(n, k), false, code, 0.f, 0.f, 0.f, nullptr,
                       nullptr, st);
  };
  auto norm = [&](const torch::Tensor& in, const torch::Tensor& res,
                  const torch::Tensor& w, const torch::Tensor& b,
                  torch::Tensor& out) {
    launch_norm_fwd(in.data_ptr(), res.data_ptr(), w.data_ptr(), b.data_ptr(),
                    out.data_ptr(), nullptr, M, H, (float)eps, false, st);
  };
  const long row = 3L * H;
  // products that take their norms along, and the attention, where a layer on
  // its own would sum in the same order
  const bool joined = norm_rows_fit(M, H) && decode_gemm_rings(M, 3 * H, H) &&
                      decode_gemm_rings(M, I, H);
  const bool attends =
      attn_rows_fit(B, S, heads, D) && decode_gemm_rings(M, H, H);
  auto norm_gemm = [&](const torch::Tensor& in, const torch::Tensor& res,
                       const torch::Tensor& w, const torch::Tensor& b,
                       torch::Tensor& normed, const torch::Tensor& W,
                       const torch::Tensor& bias, torch::Tensor& out,
                       int code) {
    if (!joined) {
      norm(in, res, w, b, normed);
      gemm(normed, W, bias, out, code);
      return;
    }
    launch_norm_rows(in.data_ptr(), res.data_ptr(), w.data_ptr(),
                     b.data_ptr(), normed.data_ptr(), (float)eps,
                     W.data_ptr(), bias.data_ptr(), out.data_ptr(), M,
                     W.size(0), H, code, st);
  };
  const float scale = (float)(1.0 / std::sqrt((double)D));
  const torch::Tensor first = aligned16(x);
  gemm(first, layers[0], layers[1], qkv, 0);
  for (size_t i = 0; i < layers.size(); i += 12) {
    const torch::Tensor* p = &layers[i];
    const char* q = (const char*)qkv.data_ptr();
    if (attends) {
      launch_attn_rows(q, mask.data_ptr<float>(), p[2].data_ptr(),
                       p[3].data_ptr(), y.data_ptr(), B, S, (int)heads, H,
                       scale, st);
    } else {
      launch_attn_fwd(q, q + 2L * H, q + 4L * H, mask.data_ptr<float>(),
                      ctx.data_ptr(), B, S, S, (int)heads, (int)heads, D,
                      false, scale, S * row, row, S * row, row, nullptr,
                      nullptr, nullptr, st);
      gemm(ctx, p[2], p[3], y, 0);
    }
    norm_gemm(y, i ? z : first, p[4], p[5], a, p[6], p[7], h, (int)act);
    gemm(h, p[8], p[9], y, 0);
    if (i + 12 < layers.size())
      norm_gemm(y, a, p[10], p[11], z, p[12], p[13], qkv, 0);
    else
      norm(y, a, p[10], p[11], z);
  }
  return z;
}
