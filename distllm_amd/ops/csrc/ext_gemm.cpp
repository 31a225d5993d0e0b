// Torch bindings of the matrix products, the hand-written MFMA GEMMs and
// hipBLASLt with a fused epilogue, and of gated units. Every model family needs these, so
// they form an extension of their own.
#include "ext_common.h"
#include "gelu_rows.h"

#include <climits>

extern "C" {
void launch_gemm_bf16(const void*, const void*, const void*, void*, int, int,
                      int, int, hipStream_t);
void launch_gemm8_bf16(const void*, const void*, const void*, void*, int, int,
                       int, int, hipStream_t);
void launch_gemm16_bf16(const void*, const void*, const void*, void*, int,
                        int, int, int, hipStream_t);
void launch_decode_gemm(const void*, const void*, const void*, void*, void*,
                        int, int, int, int, int, int, float, float, float,
                        const float*, const RowsArgs*, hipStream_t);
int decode_gemm_shares(int, int, int);
int decode_parts_shares(int, int, int);
int mid_gemm_shares(int, int, int);
void launch_norm_gemm(const void*, const void*, const void*, void*, float,
                      const void*, const void*, void*, int, int, int,
                      hipStream_t);
void launch_wide_gemm(const void*, const void*, const void*, void*, int, int,
                      int, int, float, float, float, int, hipStream_t);
int wide_gemm_tile(int, int, int, int);
void launch_clamped_glu(const void*, void*, long, int, float, float, float,
                        bool, hipStream_t);
void launch_relu2(const void*, void*, long, bool, hipStream_t);
void launch_gelu_rows(const void*, void*, long, int, const RowsArgs*, bool,
                      hipStream_t);
}

// ---- GEMM ------------------------------------------------------------------
torch::Tensor gemm_bf16(torch::Tensor A, torch::Tensor B,
                        c10::optional<torch::Tensor> bias, int64_t act) {
  CHECK_DEV(A); CHECK_CONT(A); CHECK_BF16(A);
  CHECK_DEV(B); CHECK_CONT(B); CHECK_BF16(B);
  const int M = A.size(0), K = A.size(1), N = B.size(0);
  TORCH_CHECK(B.size(1) == K, "K mismatch");
  TORCH_CHECK(M % 128 == 0 && N % 128 == 0 && K % 64 == 0,
              "gemm_bf16 requires M,N % 128 == 0 and K % 64 == 0");
  auto C = torch::empty({M, N}, A.options());
  launch_gemm_bf16(A.data_ptr(), B.data_ptr(),
                   bias ? bias->data_ptr() : nullptr, C.data_ptr(), M, N, K,
                   (int)act, cur_stream());
  return C;
}

torch::Tensor gemm8_bf16(torch::Tensor A, torch::Tensor B,
                         c10::optional<torch::Tensor> bias, int64_t act) {
  CHECK_DEV(A); CHECK_CONT(A); CHECK_BF16(A);
  CHECK_DEV(B); CHECK_CONT(B); CHECK_BF16(B);
  const int M = A.size(0), K = A.size(1), N = B.size(0);
  TORCH_CHECK(B.size(1) == K, "K mismatch");
  TORCH_CHECK(M % 256 == 0 && N % 256 == 0 && K % 64 == 0,
              "gemm8 requires M,N % 256 == 0 and K % 64 == 0");
  auto C = torch::empty({M, N}, A.options());
  launch_gemm8_bf16(A.data_ptr(), B.data_ptr(),
                    bias ? bias->data_ptr() : nullptr, C.data_ptr(), M, N, K,
                    (int)act, cur_stream());
  return C;
}

torch::Tensor gemm16_bf16(torch::Tensor A, torch::Tensor B,
                          c10::optional<torch::Tensor> bias, int64_t act) {
  CHECK_DEV(A); CHECK_CONT(A); CHECK_BF16(A);
  CHECK_DEV(B); CHECK_CONT(B); CHECK_BF16(B);
  const int M = A.size(0), K = A.size(1), N = B.size(0);
  TORCH_CHECK(B.size(1) == K, "K mismatch");
  TORCH_CHECK(M % 256 == 0 && N % 256 == 0 && K % 128 == 0,
              "gemm16 requires M,N % 256 == 0 and K % 128 == 0");
  auto C = torch::empty({M, N}, A.options());
  launch_gemm16_bf16(A.data_ptr(), B.data_ptr(),
                     bias ? bias->data_ptr() : nullptr, C.data_ptr(), M, N,
                     K, (int)act, cur_stream());
  return C;
}

static torch::Tensor decode_gemm_act(torch::Tensor X, torch::Tensor W,
                                     c10::optional<torch::Tensor> bias,
                                     int64_t splitk, int64_t act,
                                     double limit, double alpha,
                                     double shift,
                                     c10::optional<torch::Tensor> act_nums,
                                     const RowsArgs* rows,
                                     bool as_parts = false) {
  // act 1, 2 = packed gated unit (swiglu, clamped with the given constants):
  // W is [2I, K] (gate rows then up rows), output is [M, I]. act 3 = xIELU
  // with the raw numbers act_nums [2]. act 4 = GELU times a part of a table's
  // row. act 5 = relu(.)^2. act 6, 7, 8 = GELU (tanh, erf), SiLU. splitk
  // workgroups share K (activations: not 1); 0: form and split follow from
  // the sizes, as_parts: the split of decode_gemm_parts.
  CHECK_DEV(X); CHECK_CONT(X); CHECK_BF16(X);
  CHECK_DEV(W); CHECK_CONT(W); CHECK_BF16(W);
  const int M = X.size(0), K = X.size(1), N = W.size(0);
  TORCH_CHECK(W.size(1) == K, "K mismatch");
  TORCH_CHECK(M <= 256, "decode_gemm is for M <= 256");
  TORCH_CHECK(N % 64 == 0, "N % 64");
  const bool tile = splitk != 0;
  if (!tile)
    splitk = as_parts ? decode_parts_shares(M, N, K)
                      : decode_gemm_shares(M, N, K);
  TORCH_CHECK(splitk > 0 && K % (64 * splitk) == 0, "K % (64*splitk)");
  const bool glu = act == 1 || act == 2;
  TORCH_CHECK(act == 0 || !tile || splitk > 1,
              "a fused activation needs splitk > 1");
  TORCH_CHECK(!glu || N % 128 == 0, "gated-unit fusion needs N % 128 == 0");
  if (bias) {
    CHECK_DEV(bias.value()); CHECK_CONT(bias.value());
    CHECK_BF16(bias.value());
    TORCH_CHECK(bias->numel() == N, "bias must be [N]");
  }
  const float* nums = nullptr;
  if (act == 3) {
    TORCH_CHECK(act_nums.has_value() && act_nums->numel() == 2, "act_nums");
    CHECK_DEV(act_nums.value()); CHECK_F32(act_nums.value());
    nums = act_nums->data_ptr<float>();
  }
  auto out = torch::empty(
      {M, glu ? N / 2 : N},
      act == 9 ? X.options().dtype(at::kFloat) : X.options());
  if (out.numel() == 0) return out;
  X = aligned16(X);
  W = aligned16(W);
  torch::Tensor slabs;
  void* slabp = nullptr;
  if (splitk > 1) {
    slabs = torch::empty({splitk, (long)M, (long)N},
                         X.options().dtype(at::kFloat));
    slabp = slabs.data_ptr();
  }
  launch_decode_gemm(X.data_ptr(), W.data_ptr(),
                     bias ? bias->data_ptr() : nullptr, out.data_ptr(),
                     slabp, M, N, K, (int)splitk, tile, (int)act,
                     (float)limit, (float)alpha, (float)shift, nums, rows,
                     cur_stream());
  return out;
}

torch::Tensor decode_gemm(torch::Tensor X, torch::Tensor W,
                          c10::optional<torch::Tensor> bias,
                          int64_t splitk, int64_t act = 0,
                          double limit = 0.0, double alpha = 0.0,
                          double shift = 0.0,
                          c10::optional<torch::Tensor> act_nums = {}) {
  TORCH_CHECK(act >= 0 && act <= 9 && act != 4, "activation");
  return decode_gemm_act(X, W, bias, splitk, act, limit, alpha, shift,
                         act_nums, nullptr);
}

// The slabs of decode_gemm_parts, joined.
torch::Tensor decode_gemm_joined(torch::Tensor X, torch::Tensor W) {
  return decode_gemm_act(X, W, {}, 0, 0, 0., 0., 0., {}, nullptr, true);
}

// X W^T as the fp32 slabs [shares, M, N] of the workgroups that share K, for
// kernels that sum them as they read; shares > 1 (decode_parts_shares).
torch::Tensor decode_gemm_parts(torch::Tensor X, torch::Tensor W) {
  CHECK_DEV(X); CHECK_CONT(X); CHECK_BF16(X);
  CHECK_DEV(W); CHECK_CONT(W); CHECK_BF16(W);
  const int M = X.size(0), K = X.size(1), N = W.size(0);
  TORCH_CHECK(W.size(1) == K, "K mismatch");
  TORCH_CHECK(M > 0 && M <= 256 && N % 64 == 0 && K % 64 == 0, "shape");
  const int shares = decode_parts_shares(M, N, K);
  TORCH_CHECK(shares > 1, "K is not shared at this shape");
  X = aligned16(X);
  W = aligned16(W);
  auto slabs =
      torch::empty({shares, M, N}, X.options().dtype(at::kFloat));
  launch_decode_gemm(X.data_ptr(), W.data_ptr(), nullptr, nullptr,
                     slabs.data_ptr(), M, N, K, shares, false, 0, 0.f, 0.f,
                     0.f, nullptr, nullptr, cur_stream());
  return slabs;
}

// X W^T of many rows. act 0 to 3 as of the 256-row tiles (GELU by erf in 32
// bits), 4 and 5 = SwiGLU and clamped unit of packed gate and up rows; tile as
// wide_gemm_tile gives it.
torch::Tensor wide_gemm(torch::Tensor X, torch::Tensor W,
                        c10::optional<torch::Tensor> bias, int64_t act,
                        int64_t tile, double limit = 0.0, double alpha = 0.0,
                        double shift = 0.0) {
  CHECK_DEV(X); CHECK_CONT(X); CHECK_BF16(X);
  CHECK_DEV(W); CHECK_CONT(W); CHECK_BF16(W);
  TORCH_CHECK(X.dim() == 2 && W.dim() == 2 && W.size(1) == X.size(1) &&
                  X.device() == W.device(),
              "operands");
  const int64_t M = X.size(0), K = X.size(1), N = W.size(0);
  TORCH_CHECK(M > 0 && M < 1 << 30 && N > 0 && N % 256 == 0 && K % 64 == 0 &&
                  K >= 128 && N * K < 1L << 30,
              "wide_gemm: sizes");
  TORCH_CHECK(act >= 0 && act <= 5 && tile >= 4 && tile <= 8, "wide_gemm");
  const int64_t rows = (M + 32 * tile - 1) / (32 * tile);
  TORCH_CHECK(rows * (N / 256) * (N / 256) * 8 < 1L << 32,
              "wide_gemm: too many tiles");
  const c10::DeviceGuard guard(X.device());
  if (bias) {
    CHECK_DEV(bias.value()); CHECK_CONT(bias.value());
    CHECK_BF16(bias.value());
    TORCH_CHECK(bias->numel() == N && bias->device() == X.device(),
                "bias must be [N]");
    bias = aligned16(bias.value());
  }
  auto out = torch::empty({M, act >= 4 ? N / 2 : N}, X.options());
  X = aligned16(X);
  W = aligned16(W);
  launch_wide_gemm(X.data_ptr(), W.data_ptr(),
                   bias ? bias->data_ptr() : nullptr, out.data_ptr(), (int)M,
                   (int)N, (int)K, (int)act, (float)limit, (float)alpha,
                   (float)shift, (int)tile, cur_stream());
  return out;
}

// X W^T of 65 rows and more by tiles of 64 x 64; shares as mid_gemm_shares
// gives them; act 0, 6, 7, 8 as of decode_gemm.
torch::Tensor mid_gemm(torch::Tensor X, torch::Tensor W,
                       c10::optional<torch::Tensor> bias, int64_t shares,
                       int64_t act) {
  CHECK_DEV(X); CHECK_CONT(X); CHECK_BF16(X);
  CHECK_DEV(W); CHECK_CONT(W); CHECK_BF16(W);
  TORCH_CHECK(X.dim() == 2 && W.dim() == 2 && W.size(1) == X.size(1) &&
                  X.device() == W.device(),
              "operands");
  const int64_t M = X.size(0), K = X.size(1), N = W.size(0);
  TORCH_CHECK(M > 0 && N > 0 && N % 64 == 0 && K >= 128 && shares >= 1 &&
                  shares <= 4 && K % (64 * shares) == 0 &&
                  M * N < 1L << 30,
              "mid_gemm: sizes");
  TORCH_CHECK(act == 0 || (act >= 6 && act <= 8), "activation");
  const c10::DeviceGuard guard(X.device());
  if (bias) {
    CHECK_DEV(bias.value()); CHECK_CONT(bias.value());
    CHECK_BF16(bias.value());
    TORCH_CHECK(bias->numel() == N && bias->device() == X.device(),
                "bias must be [N]");
  }
  auto out = torch::empty({M, N}, X.options());
  X = aligned16(X);
  W = aligned16(W);
  torch::Tensor slabs;
  if (shares > 1)
    slabs = torch::empty({shares, M, N}, X.options().dtype(at::kFloat));
  launch_decode_gemm(X.data_ptr(), W.data_ptr(),
                     bias ? bias->data_ptr() : nullptr, out.data_ptr(),
                     shares > 1 ? slabs.data_ptr() : nullptr, (int)M, (int)N,
                     (int)K, (int)shares, 64, (int)act, 0.f, 0.f, 0.f, nullptr,
                     nullptr, cur_stream());
  return out;
}

// x = a + b, one row, and the product of its RMS norm (act 1: gated unit)
std::vector<torch::Tensor> norm_gemm(torch::Tensor a, torch::Tensor b,
                                     torch::Tensor w_norm, double eps,
                                     torch::Tensor W,
                                     c10::optional<torch::Tensor> bias,
                                     int64_t act) {
  for (const auto& t : {a, b, w_norm, W}) {
    CHECK_DEV(t); CHECK_CONT(t); CHECK_BF16(t);
    TORCH_CHECK((uintptr_t)t.data_ptr() % 16 == 0, "16-byte alignment");
  }
  TORCH_CHECK(W.dim() == 2, "W");
  const int K = W.size(1), N = W.size(0);
  TORCH_CHECK(K % 64 == 0 && K >= 1280 && K <= 8192 && a.numel() == K &&
                  b.numel() == K && w_norm.numel() == K,
              "norm_gemm: one row of 1280 to 8192 numbers");
  TORCH_CHECK(act == 0 || act == 1 || act == 9, "activation");
  TORCH_CHECK(N > 0 && N % (act == 1 ? 128 : 64) == 0, "columns");
  if (bias) {
    CHECK_DEV(bias.value()); CHECK_CONT(bias.value());
    CHECK_BF16(bias.value());
    TORCH_CHECK(bias->numel() == N, "bias");
  }
  auto out = torch::empty(
      {1, act == 1 ? N / 2 : N},
      act == 9 ? a.options().dtype(at::kFloat) : a.options());
  auto sum = torch::empty_like(b);
  launch_norm_gemm(a.data_ptr(), b.data_ptr(), w_norm.data_ptr(),
                   sum.data_ptr(), (float)eps, W.data_ptr(),
                   bias ? bias->data_ptr() : nullptr, out.data_ptr(), N, K,
                   (int)act, cur_stream());
  return {out, sum};
}

static RowsArgs rows_args(const torch::Tensor& tokens,
                          const torch::Tensor& table, long M, int64_t col0,
                          int64_t n, long N) {
  CHECK_DEV(tokens); CHECK_CONT(tokens);
  CHECK_DEV(table); CHECK_CONT(table); CHECK_T(table);
  TORCH_CHECK(tokens.scalar_type() == at::kLong && tokens.numel() == M,
              "tokens must be int64, one per row");
  TORCH_CHECK(table.dim() == 2 && n > 0 && n <= N && col0 >= 0 &&
                  col0 + n <= table.size(1),
              "table columns");
  return {(const long*)tokens.data_ptr<int64_t>(), table.data_ptr(),
          (long)table.size(1), (int)col0, (int)n};
}

// gelu(X W^T) * table[token, col0 : col0 + n], zeros in the other columns
torch::Tensor decode_gemm_rows(torch::Tensor X, torch::Tensor W,
                               int64_t splitk, torch::Tensor tokens,
                               torch::Tensor table, int64_t col0, int64_t n) {
  CHECK_SAME(X, table);
  const RowsArgs r =
      rows_args(tokens, table, X.size(0), col0, n, W.size(0));
  return decode_gemm_act(X, W, {}, splitk, 4, 0., 0., 0., {}, &r);
}

torch::Tensor gelu_rows(torch::Tensor z, torch::Tensor tokens,
                        torch::Tensor table, int64_t col0, int64_t n) {
  CHECK_DEV(z); CHECK_CONT(z); CHECK_T(z); CHECK_SAME(z, table);
  TORCH_CHECK(z.dim() == 2 && z.size(1) % 8 == 0, "columns % 8");
  const long M = z.size(0);
  const int N = z.size(1);
  const RowsArgs r = rows_args(tokens, table, M, col0, n, N);
  auto out = torch::empty_like(z);
  if (M > 0)
    launch_gelu_rows(z.data_ptr(), out.data_ptr(), M, N, &r, is_f32(z),
                     cur_stream());
  return out;
}

torch::Tensor clamped_glu(torch::Tensor gu, double limit, double alpha,
                          double shift) {
  CHECK_DEV(gu); CHECK_CONT(gu); CHECK_T(gu);
  const long R = gu.size(0);
  const int F = gu.size(1) / 2;
  TORCH_CHECK(gu.dim() == 2 && F % 8 == 0, "halves must be % 8");
  auto out = torch::empty({R, F}, gu.options());
  if (R > 0)
    launch_clamped_glu(gu.data_ptr(), out.data_ptr(), R, F, (float)limit,
                       (float)alpha, (float)shift, is_f32(gu), cur_stream());
  return out;
}

torch::Tensor relu2(torch::Tensor z) {
  CHECK_DEV(z); CHECK_CONT(z); CHECK_T(z);
  TORCH_CHECK(z.numel() % 8 == 0, "size % 8");
  auto out = torch::empty_like(z);
  if (z.numel() > 0)
    launch_relu2(z.data_ptr(), out.data_ptr(), z.numel(), is_f32(z),
                 cur_stream());
  return out;
}

// blt_gemm.cpp: hipBLASLt GEMM with fused bias/GELU/swish epilogue.
torch::Tensor blt_linear(torch::Tensor x, torch::Tensor w,
                         c10::optional<torch::Tensor> bias, int64_t epi);

// What a decode step of a captured batch reads, from lists into tensors of the host:
// tokens (64 bits), lengths, slots of states (of no rows where there are none), block
// table. Rows past those that are there have length 1 and otherwise zeros.
static void step_inputs(torch::Tensor to_tokens, torch::Tensor to_lengths,
                        torch::Tensor to_slots, torch::Tensor table,
                        const py::list& tokens, const py::list& lengths,
                        const py::list& slots, const py::list& blocks) {
  const int64_t n = (int64_t)tokens.size(), batch = to_tokens.numel();
  const bool states = to_slots.numel() > 0;
  for (const auto& t : {to_tokens, to_lengths, to_slots, table})
    TORCH_CHECK(t.device().is_cpu() && t.is_contiguous() &&
                    (t.scalar_type() == at::kInt || t.is_same(to_tokens)),
                "step_inputs: int32 tensors of the host");
  TORCH_CHECK(to_tokens.scalar_type() == at::kLong &&
                  to_lengths.numel() == batch && table.dim() == 2 &&
                  table.size(0) == batch &&
                  (!states || to_slots.numel() == batch),
              "step_inputs: tensors of one batch");
  TORCH_CHECK(n <= batch && (int64_t)lengths.size() == n &&
                  (int64_t)blocks.size() == n &&
                  (int64_t)slots.size() == (states ? n : 0),
              "step_inputs: a row each");
  auto number = [](PyObject* o) {
    const long v = PyLong_AsLong(o);
    if (v == -1 && PyErr_Occurred()) throw py::error_already_set();
    return v;
  };
  auto word = [&](PyObject* o) {
    const long v = number(o);
    TORCH_CHECK(v >= INT_MIN && v <= INT_MAX, "step_inputs: 32 bits");
    return (int)v;
  };
  const int64_t width = table.size(1);
  int64_t* token = to_tokens.data_ptr<int64_t>();
  int* length = to_lengths.data_ptr<int>();
  int* slot = states ? to_slots.data_ptr<int>() : nullptr;
  int* to = width > 0 ? table.data_ptr<int>() : nullptr;
  for (int64_t i = 0; i < batch; ++i, to += width) {
    token[i] = i < n ? number(tokens[i].ptr()) : 0;
    length[i] = i < n ? word(lengths[i].ptr()) : 1;
    if (states) slot[i] = i < n ? word(slots[i].ptr()) : 0;
    int64_t k = 0;
    if (i < n) {
      const auto row = py::reinterpret_steal<py::object>(
          PySequence_Fast(blocks[i].ptr(), "step_inputs: blocks"));
      if (!row) throw py::error_already_set();
      k = PySequence_Fast_GET_SIZE(row.ptr());
      TORCH_CHECK(k <= width, "step_inputs: a row of ", k, " blocks of ",
                  width);
      PyObject** items = PySequence_Fast_ITEMS(row.ptr());
      for (int64_t j = 0; j < k; ++j) to[j] = word(items[j]);
    }
    std::fill(to + k, to + width, 0);
  }
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("blt_linear", &blt_linear,
        "hipBLASLt linear with fused bias/GELU/swish epilogue");
  m.def("gemm_bf16", &gemm_bf16);
  m.def("gemm8_bf16", &gemm8_bf16);
  m.def("gemm16_bf16", &gemm16_bf16);
  m.def("decode_gemm", &decode_gemm, py::arg("X"), py::arg("W"),
        py::arg("bias"), py::arg("splitk"), py::arg("act") = 0,
        py::arg("limit") = 0.0, py::arg("alpha") = 0.0,
        py::arg("shift") = 0.0, py::arg("act_nums") = py::none());
  m.def("wide_gemm", &wide_gemm, py::arg("X"), py::arg("W"), py::arg("bias"),
        py::arg("act"), py::arg("tile"), py::arg("limit") = 0.0,
        py::arg("alpha") = 0.0, py::arg("shift") = 0.0);
  m.def("wide_gemm_tile", &wide_gemm_tile);
  m.def("mid_gemm", &mid_gemm);
  m.def("mid_gemm_shares", &mid_gemm_shares);
  m.def("norm_gemm", &norm_gemm);
  m.def("decode_gemm_parts", &decode_gemm_parts);
  m.def("decode_gemm_joined", &decode_gemm_joined);
  m.def("decode_gemm_shares", &decode_gemm_shares);
  m.def("decode_parts_shares", &decode_parts_shares);
  m.def("decode_gemm_rows", &decode_gemm_rows);
  m.def("gelu_rows", &gelu_rows);
  m.def("clamped_glu", &clamped_glu);
  m.def("relu2", &relu2);
  m.def("step_inputs", &step_inputs);
}
