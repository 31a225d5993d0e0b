"""Op dispatch layer: hand-written HIP kernels on GPU, fp32 torch
reference on CPU.

Policy (required by the build rules): on a GPU tensor the HIP extension
is the ONLY path — if its module failed to import, GPU calls raise
immediately instead of silently falling back to eager PyTorch. CPU
tensors use distllm_amd.ops.torch_ref (fp32), which also serves as the
numerics ground truth in tests.
"""

from __future__ import annotations

import math
import os
from typing import NamedTuple

import torch
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

from . import torch_ref
from .native import Native

# One namespace over the built extension modules (native.py).
_hip_ops = Native()
HAVE_HIP = not _hip_ops.errors
_HIP_ERR: Exception | None = next(iter(_hip_ops.errors.values()), None)


def _require_hip(name: str = "_hip_ops"):
    _hip_ops.require(name)


# Activation codes shared with csrc/gemm.hip
ACT_NONE, ACT_GELU_TANH, ACT_GELU_ERF, ACT_SILU = 0, 1, 2, 3


def norm_fwd(x, res=None, w=None, b=None, eps=1e-5, rms=False):
    if x.is_cuda:
        _require_hip()
        return _hip_ops.norm_fwd(x, res, w, b, None, eps, rms)
    return torch_ref.norm_fwd(x, res, w, b, eps, rms)


def norm_fwd_sum(x, res, w, b=None, eps=1e-5, rms=False):
    """Fused (x+res) -> norm; returns (normed, x+res). Replaces the
    separate residual-add elementwise pass in pre-norm decoders."""
    if x.is_cuda:
        _require_hip()
        summed = torch.empty_like(x)
        out = _hip_ops.norm_fwd(x, res, w, b, summed, eps, rms)
        return out, summed
    return torch_ref.norm_fwd(x, res, w, b, eps, rms, return_sum=True)


def norm_parts_sum(x, res, w, eps=1e-5):
    """norm_fwd_sum (RMS) of what linear_parts returned."""
    if x.dtype == torch.float32 and x.is_cuda:
        return _hip_ops.norm_parts(x, res, w, eps)
    return norm_fwd_sum(x.view(res.shape), res, w, eps=eps, rms=True)


def layer_norm(x, w, b, eps=1e-12, res=None):
    return norm_fwd(x, res=res, w=w, b=b, eps=eps, rms=False)


def rms_norm(x, w, eps=1e-5, res=None):
    return norm_fwd(x, res=res, w=w, b=None, eps=eps, rms=True)


def bias_gelu(x, bias=None, erf=False):
    if x.is_cuda:
        _require_hip()
        return _hip_ops.bias_gelu(x, bias, erf)
    return torch_ref.bias_gelu(x, bias, erf)


def swiglu(gate, up):
    if gate.is_cuda:
        _require_hip()
        return _hip_ops.swiglu(gate.contiguous(), up.contiguous())
    return torch_ref.swiglu(gate, up)


def bias_add(x, bias):
    if x.is_cuda:
        _require_hip()
        return _hip_ops.bias_add(x, bias)
    return torch_ref.bias_add(x, bias)


def mean_pool(hidden, mask, normalize=False):
    mask = mask.int()
    if hidden.is_cuda:
        _require_hip()
        return _hip_ops.mean_pool(hidden.contiguous(), mask.contiguous(),
                                  normalize)
    return torch_ref.mean_pool(hidden, mask, normalize)


def last_token_pool(hidden, mask, left_padded=False, normalize=False):
    mask = mask.int()
    if hidden.is_cuda:
        _require_hip()
        return _hip_ops.last_token_pool(hidden.contiguous(), mask.contiguous(),
                                        left_padded, normalize)
    return torch_ref.last_token_pool(hidden, mask, left_padded, normalize)


def l2_normalize(x):
    if x.is_cuda:
        _require_hip()
        return _hip_ops.l2_normalize(x.float().contiguous())
    return torch_ref.l2_normalize(x)


def adjacent_cosine(emb):
    if emb.is_cuda:
        _require_hip()
        return _hip_ops.adjacent_cosine(emb.float().contiguous())
    return torch_ref.adjacent_cosine(emb)


def gemm(A, B, bias=None, act=ACT_NONE):
    """C = A @ B^T via the hand-written MFMA kernel (GPU, padded shapes)
    or fp32 reference (CPU)."""
    if A.is_cuda:
        _require_hip("_hip_gemm")
        return _hip_ops.gemm_bf16(A, B, bias, act)
    return torch_ref.gemm(A, B, bias, act)


_GEMM_CHOICE: dict[tuple, str] = {}


def _blaslt_path(x2, weight, bias, act):
    out = torch.nn.functional.linear(x2, weight, bias)
    if act == ACT_GELU_TANH:
        out = bias_gelu(out, None, erf=False)
    elif act == ACT_GELU_ERF:
        out = bias_gelu(out, None, erf=True)
    elif act == ACT_SILU:
        out = (
            torch.nn.functional.silu(out.float()).to(out.dtype)
            if not out.is_cuda else _silu_gpu(out)
        )
    return out


def _blt_fused_path(x2, weight, bias, act):
    """ONE hipBLASLt call with the bias/GELU/swish applied in the GEMM
    epilogue — no separate elementwise pass over the [M, N] output."""
    epi = (1 if act in (ACT_GELU_TANH, ACT_GELU_ERF)
           else 2 if act == ACT_SILU else 0)
    return _hip_ops.blt_linear(x2, weight, bias, epi)


def _autotune_gemm(x2, weight, bias, act):
    """Measure hipBLASLt(+epilogue kernel) vs hipBLASLt-fused-epilogue
    vs the fused gemm8 MFMA kernel once per (M-bucket, N, K, act) and
    cache the winner."""
    import time as _t

    def timeit(fn):
        try:
            fn()
        except RuntimeError:
            return float("inf")
        torch.cuda.synchronize()
        t0 = _t.perf_counter()
        for _ in range(5):
            fn()
        torch.cuda.synchronize()
        return _t.perf_counter() - t0

    times = {
        "blaslt": timeit(lambda: _blaslt_path(x2, weight, bias, act)),
        "gemm8": timeit(lambda: _hip_ops.gemm8_bf16(x2, weight, bias, act)),
        "blt_fused": timeit(lambda: _blt_fused_path(x2, weight, bias, act)),
    }
    if x2.shape[1] % 128 == 0:  # gemm16 needs K % 128 == 0
        times["gemm16"] = timeit(
            lambda: _hip_ops.gemm16_bf16(x2, weight, bias, act))
    return min(times, key=times.get)


# activation codes of decode_gemm for those of linear
_DECODE_ACT = {ACT_NONE: 0, ACT_GELU_TANH: 6, ACT_GELU_ERF: 7, ACT_SILU: 8}


def _few_rows(x2, weight, bias=None, columns=64):
    """Whether a product of x2 with the rows of weight (in multiples of
    `columns`) and an activation in the same launch takes decode_gemm
    (csrc/decode_gemm.hip). Up to 64 rows: measured against the library's
    product, 64 rows of 28672 x 4096, gated, 51 and 57 us, of 768 x 768 3.8 and
    7; the slowest gated one of 14 sizes is 16384 x 8192 (61 and 56). Up to 256
    rows of up to 16384 columns, in which gate and up-projection reach the
    activation in 32 bits: against the library's product and the unit as a
    launch of its own, which round them to 16 in between, 128 rows of 16384 x
    1024 9.8 and 14, of 8192 x 2048 14 and 16, of 4096 x 1024 10.6 and 11.8, of
    2048 x 1024 9.1 and 8.1; 256 rows 13.7 and 19, 21 and 23, 15 and 11.7, 12.5
    and 11.1. Wider ones are the library's above 64 rows (28672 x 4096, 128 rows:
    64 and 58). K of a single 64-wide chunk, which would leave three of a
    workgroup's four waves idle, keeps its general path."""
    M, K = x2.shape
    N = weight.shape[0]
    return ((M <= 64 or (M <= 256 and N <= 16384))
            and K % 64 == 0 and K >= 128 and N % columns == 0 and N > 0
            and x2.dtype == weight.dtype == torch.bfloat16
            and x2.is_contiguous() and weight.is_contiguous()
            and x2.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0
            and (bias is None or (bias.dtype == torch.bfloat16
                                  and bias.shape == (N,)
                                  and bias.is_contiguous())))


# values of DISTLLM_GEMM that ask for another form than that of few rows
_OTHER_FORMS = ("blaslt", "gemm8", "gemm16")


def _wide_logits(M, N, K) -> bool:
    """Columns of a vocabulary, for which decode_gemm and the library take
    turns from 17 rows on (64 rows, us: 151936 x 4096 269 and 237, 128256 x
    4096 223 and 200, 250000 x 1536 176 and 161, 151936 x 2048 139 and 152): the
    choice is measured."""
    return M > 16 and N > 32768 and K >= 1536


# sizes (M, N, K, bias or not) of products that ran with their measured choice
# and have another form to go by
_WIDE_RUN: set[tuple] = set()


def _measurable(M, N, K, bias) -> bool:
    """While a graph is captured nothing can be measured, neither the choice
    nor the library's algorithm for a new M: only sizes that ran before go by
    the measured choice."""
    return ((M, N, K, bias is not None) in _WIDE_RUN
            or not torch.cuda.is_current_stream_capturing())


def _to_choose(M, N, K, bias) -> bool:
    """Whether a product of up to 64 rows goes by the measured choice."""
    return _wide_logits(M, N, K) and _measurable(M, N, K, bias)


def _gemm_mode() -> str:
    return os.environ.get("DISTLLM_GEMM", "auto")


# what _recorded asks in every call, found once
_grad_enabled, _autocast = torch.is_grad_enabled, torch.is_autocast_enabled
_tracing, _function_modes = torch._C._is_tracing, torch._C._len_torch_function_stack
_dispatch_modes = torch._C._len_torch_dispatch_stack
_transforms = torch._C._functorch.peek_interpreter_stack
_PLAIN = (torch.Tensor, torch.nn.Parameter)


def _recorded(*tensors) -> bool:
    """Whether something follows these tensors that a native kernel would
    pass by: gradients, transforms, traces, modes of dispatch or of functions
    (but for the one of a default device), tensors of another make, a cast to
    another 16-bit type."""
    if (_dispatch_modes() or _transforms() is not None
            or torch.autograd.forward_ad._current_level >= 0 or _tracing()
            or (_function_modes()
                and any(type(m) is not DeviceContext
                        for m in _get_current_function_mode_stack()))
            or (_autocast()
                and torch.get_autocast_dtype("cuda") != torch.bfloat16)):
        return True
    grad = _grad_enabled()
    for t in tensors:
        if t is not None and (type(t) not in _PLAIN
                              or (grad and t.requires_grad)):
            return True
    return False


# activation codes of wide_gemm behind those of linear
_WIDE_SWIGLU, _WIDE_CLAMPED = 4, 5


def _own_product(x2, weight, bias) -> bool:
    """Whether the operands are as mid_gemm and wide_gemm take them and nothing
    asks for another product."""
    return (x2.dtype == weight.dtype == torch.bfloat16
            and x2.is_contiguous() and weight.is_contiguous()
            and x2.device == weight.device
            and (bias is None or (
                bias.dtype == torch.bfloat16
                and bias.shape == weight.shape[:1]
                and bias.is_contiguous() and bias.device == x2.device))
            and _gemm_mode() not in _OTHER_FORMS
            and not _recorded(x2, weight, bias))


def _mid_shares(x2, weight, bias) -> int:
    """The shares of K with which x2 @ weight^T goes by csrc/decode_gemm.hip's
    blocks of 64 rows, 0 where it does not (mid_gemm_shares there has the
    measurements)."""
    M, K = x2.shape
    N = weight.shape[0]
    if M <= 64 or M * N > 512 * 4096:  # tiles of 64 x 64
        return 0
    shares = _hip_ops.mid_gemm_shares(M, N, K)
    return shares if shares and _own_product(x2, weight, bias) else 0


def _wide_tile(x2, weight, bias, act) -> int:
    """The tile with which x2 @ weight^T, bias and activation or gated unit go
    in one launch of csrc/wide_gemm.hip, 0 where another way is faster (the
    measurements are there, at wide_gemm_tile) or has to be taken."""
    M, K = x2.shape
    N = weight.shape[0]
    if (M <= 64 or M * N < 96 * 127 * 256  # its least tiles
            or (act == ACT_NONE and M <= 256)):
        return 0
    tile = _hip_ops.wide_gemm_tile(M, N, K, act)
    return tile if tile and _own_product(x2, weight, bias) else 0


def linear(x, weight, bias=None, act=ACT_NONE):
    """Linear layer entry used by models. GPU path: the products of few rows
    (decode_gemm.hip, with the activation) for M <= 64 (_few_rows) and, by
    blocks of them, where _mid_shares says so, those of many rows
    (wide_gemm.hip, with the activation) where _wide_tile says so;
    else an autotuned choice between hipBLASLt (plain and fused-epilogue), the
    other hand-written MFMA GEMMs (gemm8.hip, 8-phase gemm16.hip) and, for M
    <= 256, decode_gemm.hip and blocks that share K. Override with
    DISTLLM_GEMM=blaslt|gemm8|gemm16|decode (the last for M <= 256, gemm8 and
    gemm16 at their multiples of 256 rows; without an activation M <= 256
    stays a choice for those two, at other sizes they mean the library)."""
    orig_shape = x.shape
    x2 = x.reshape(-1, orig_shape[-1])
    M, K = x2.shape
    N = weight.shape[0]
    if x.is_cuda:
        _require_hip("_hip_gemm")
        mode = _gemm_mode()
        if x2.dtype == torch.float32:  # true 32-bit products
            mode = "blaslt"
        if (mode not in _OTHER_FORMS and M <= 64
                and not (act == ACT_NONE and _to_choose(M, N, K, bias))
                and _few_rows(x2, weight, bias)):
            out = _hip_ops.decode_gemm(x2, weight, bias, 0, _DECODE_ACT[act])
            return out.reshape(*orig_shape[:-1], N)
        asked = mode == "decode" and M <= 256  # for that form alone
        shares = 0 if asked else _mid_shares(x2, weight, bias)
        # up to 256 rows whose K is shared, a second launch, it is one of the
        # measured choices: us in a graph, this and decode_gemm, 80 rows of 4096 x
        # 4096 16.4 and 15.4, of 2048 x 8192 16.6 and 17.0, of 768 x 3072 9.6 and
        # 10.7, 160 rows 10.2 and 12.9 (and the library's 9.6)
        if shares and not (shares > 1 and act == ACT_NONE and M <= 256
                           and _measurable(M, N, K, bias)):
            return _hip_ops.mid_gemm(x2, weight, bias, shares,
                                     _DECODE_ACT[act]).view(
                *orig_shape[:-1], N)
        tile = 0 if asked else _wide_tile(x2, weight, bias, act)
        if tile:
            return _hip_ops.wide_gemm(x2, weight, bias, act, tile).view(
                *orig_shape[:-1], N)
        if (mode != "blaslt" and act == ACT_NONE and M <= 256
                and N % 64 == 0 and K % 64 == 0 and x2.is_contiguous()
                and (bias is None or bias.shape == (N,))):
            if mode == "decode":  # forced in-chain A/B (profiling)
                out = _hip_ops.decode_gemm(x2, weight, bias, 0)
                return out.reshape(*orig_shape[:-1], N)
            # bucket by padded M so varying decode/prefill
            # batch sizes reuse one tuning decision
            key = ("dec", 128 if M <= 128 else 256, N, K,
                   bias is not None) + (("mid",) if shares else ())
            choice = _GEMM_CHOICE.get(key)
            if choice is None:
                import time as _t

                def timeit(fn):
                    fn()
                    torch.cuda.synchronize()
                    t0 = _t.perf_counter()
                    for _ in range(10):
                        fn()
                    torch.cuda.synchronize()
                    return _t.perf_counter() - t0

                times = {
                    "blaslt": timeit(lambda: torch.nn.functional.linear(
                        x2, weight, bias)),
                    "decode": timeit(lambda: _hip_ops.decode_gemm(
                        x2, weight, bias, 0)),
                }
                if shares:
                    times["mid"] = timeit(lambda: _hip_ops.mid_gemm(
                        x2, weight, bias, shares, 0))
                try:  # hipBLASLt with measured algo search (blt_gemm.cpp)
                    times["blt_fused"] = timeit(
                        lambda: _blt_fused_path(x2, weight, bias, act))
                except RuntimeError:
                    pass
                choice = min(times, key=times.get)
                _GEMM_CHOICE[key] = choice
            if choice == "decode":
                out = _hip_ops.decode_gemm(x2, weight, bias, 0)
            elif choice == "mid":
                out = _hip_ops.mid_gemm(x2, weight, bias, shares, 0)
            elif choice == "blt_fused":
                out = _blt_fused_path(x2, weight, bias, act)
            else:
                out = torch.nn.functional.linear(x2, weight, bias)
            if shares or (M <= 64 and _wide_logits(M, N, K)):
                _WIDE_RUN.add((M, N, K, bias is not None))
            return out.reshape(*orig_shape[:-1], N)
        shapes_ok = (M % 256 == 0 and N % 256 == 0 and K % 64 == 0
                     and x2.is_contiguous())
        if shapes_ok and mode != "blaslt":
            if mode == "gemm8":
                out = _hip_ops.gemm8_bf16(x2, weight, bias, act)
            elif mode == "gemm16":
                out = _hip_ops.gemm16_bf16(x2, weight, bias, act)
            else:  # auto
                # coarse bucket above 16k rows: packed varlen batches
                # produce a different M per batch, and a fresh
                # 4-implementation autotune probe per distinct M
                # (~100ms each) dominated the semantic-chunk pipeline
                key = ("big" if M >= 16384 else M // 4096, N, K, act)
                choice = _GEMM_CHOICE.get(key)
                if choice is None:
                    choice = _autotune_gemm(x2, weight, bias, act)
                    _GEMM_CHOICE[key] = choice
                if choice == "gemm8":
                    out = _hip_ops.gemm8_bf16(x2, weight, bias, act)
                elif choice == "gemm16":
                    out = _hip_ops.gemm16_bf16(x2, weight, bias, act)
                elif choice == "blt_fused":
                    out = _blt_fused_path(x2, weight, bias, act)
                else:
                    out = _blaslt_path(x2, weight, bias, act)
        else:
            out = _blaslt_path(x2, weight, bias, act)
    else:
        out = _blaslt_path(x2, weight, bias, act)
    return out.reshape(*orig_shape[:-1], N)


# decode_gemm's code for linear(...).float()
_DECODE_F32 = 9
_LINEAR = linear


def linear_f32(x, weight):
    """linear(x, weight).float(). Up to 64 rows that take decode_gemm are stored as
    32 bits by the product, without a launch of 4 to 5 us that widens them, unless
    ops.linear has been replaced and is to see every product."""
    x2 = x.reshape(-1, x.shape[-1])
    M, K = x2.shape
    N = weight.shape[0]
    if (x.is_cuda and M <= 64 and x2.dtype == torch.bfloat16
            and linear is _LINEAR and _gemm_mode() not in _OTHER_FORMS
            and not _to_choose(M, N, K, None) and _few_rows(x2, weight)
            and not _recorded(x2, weight)):
        _require_hip("_hip_gemm")
        return _hip_ops.decode_gemm(x2, weight, None, 0, _DECODE_F32).reshape(
            *x.shape[:-1], N)
    return linear(x, weight).float()


def linear_parts(x, weight, bias=None):
    """linear, for a consumer that can sum: where few rows share K among
    workgroups (17 to 64 rows, csrc/decode_gemm.hip), the fp32 slabs
    [shares, M, N] without their sum and without the bias, which saves the
    summing launch; else linear's output [M, N]."""
    x2 = x.reshape(-1, x.shape[-1])
    M, K = x2.shape
    if (x.is_cuda and 0 < M <= 64
            and _gemm_mode() not in _OTHER_FORMS):
        _require_hip("_hip_gemm")
        if (_few_rows(x2, weight, bias)
                and _hip_ops.decode_parts_shares(M, weight.shape[0], K) > 1):
            return _hip_ops.decode_gemm_parts(x2, weight)
    return linear(x2, weight, bias)


def linear_joined(x, weight):
    """linear, whose sums are those of linear_parts' slabs in every bit: for a
    consumer that wants [M, N] where another of the same numbers takes slabs (of
    17 to 32 rows linear may be another split of K)."""
    x2 = x.reshape(-1, x.shape[-1])
    M, K = x2.shape
    if x.is_cuda and 0 < M <= 64 and _gemm_mode() not in _OTHER_FORMS:
        _require_hip("_hip_gemm")
        if (_few_rows(x2, weight)
                and _hip_ops.decode_parts_shares(M, weight.shape[0], K) > 1):
            return _hip_ops.decode_gemm_joined(x2, weight)
    return linear(x2, weight)


def _norm_in_product(a, b, w_norm, weight, least):
    """Whether a + b is one row whose norm the product of it with `weight`
    takes into its launch (csrc/norm_row.h): up to 8192 columns, at least
    `least`, so that every wave has five chunks. Two rows already cost every
    workgroup more than the launch saves."""
    K = weight.shape[1]
    return (a.is_cuda and a.numel() == b.numel() == K
            and a.shape[-1] == b.shape[-1] == K
            and least <= K <= 8192
            and a.dtype == b.dtype == w_norm.dtype == torch.bfloat16
            and all(t.is_contiguous() and t.data_ptr() % 16 == 0
                    for t in (a, b, w_norm, weight)))


def norm_linear(a, b, w_norm, eps, weight, bias=None, gated=False,
                shares=False, f32=False):
    """x = a + b, and the linear (or, gated, the SwiGLU of the packed gate and
    up rows) of its RMS norm times w_norm -> (linear [M, N], x like b); a may
    be what linear_parts returned, and with `shares` the linear is of that
    kind; with `f32` (no bias) it is linear_f32. One row is one launch."""
    N = weight.shape[0]
    if (_gemm_mode() not in _OTHER_FORMS and not (f32 and linear is not _LINEAR)
            and weight.dtype == torch.bfloat16 and weight.shape[1] % 64 == 0
            and N % (128 if gated else 64) == 0
            and (bias is None or (bias.dtype == torch.bfloat16
                                  and bias.shape == (N,)
                                  and bias.is_contiguous()))
            and _norm_in_product(a, b, w_norm, weight, 1280)):
        _require_hip("_hip_gemm")
        return tuple(_hip_ops.norm_gemm(a, b, w_norm, eps, weight, bias,
                                        _DECODE_F32 if f32 else int(gated)))
    h, x = norm_parts_sum(a, b, w_norm, eps=eps)
    h = h.reshape(-1, h.shape[-1])
    if gated:
        return gateup_swiglu(h, weight, bias), x
    if f32:
        return linear_f32(h, weight), x
    return (linear_parts if shares else linear)(h, weight, bias), x


def norm_linear_fp8(a, b, w_norm, eps, wq, scale, bias=None, gated=False):
    """norm_linear on weights quantized as for gemv_fp8 (but for the few
    columns of a long K that gemv_fp8 takes by column)."""
    N, K = wq.shape
    if (K % 128 == 0 and (gated or N > 512 or K < 4096)
            and _norm_in_product(a, b, w_norm, wq, 2560)):
        _require_hip()
        return tuple(_hip_ops.gemv_fp8_norm(a, b, w_norm, eps, wq, scale,
                                            bias, gated))
    h, x = norm_parts_sum(a, b, w_norm, eps=eps)
    h = h.reshape(-1, h.shape[-1])
    if gated:
        return gateup_swiglu_fp8(h, wq, scale, bias), x
    return gemv_fp8(h, wq, scale, bias), x


def _silu_gpu(x):
    # standalone silu via the swiglu kernel with up=1 is wasteful; use a
    # dedicated path: silu(x) = swiglu(x, ones) avoided — bias_gelu
    # kernel family does not cover silu alone, so fall back to torch for
    # this rare case (plain silu without mul is not on any hot path).
    return torch.nn.functional.silu(x)


def attn_fwd(Q, K, V, mask=None, causal=False, scale=None):
    D = Q.shape[-1]
    if scale is None:
        scale = 1.0 / math.sqrt(D)
    if Q.is_cuda:
        _require_hip()
        if D not in (64, 128):
            # head_dim not natively tiled (e.g. small ESM2 variants,
            # D=16/24/32/96): zero-pad to the next native width — exact,
            # since padded dims add 0 to QK^T and produce 0 in O.
            Dp = 64 if D < 64 else 128
            pad = Dp - D
            Qp = torch.nn.functional.pad(Q, (0, pad))
            Kp = torch.nn.functional.pad(K, (0, pad))
            Vp = torch.nn.functional.pad(V, (0, pad))
            O = _hip_ops.attn_fwd(
                Qp, Kp, Vp,
                mask.contiguous() if mask is not None else None,
                causal, scale,
            )
            return O[..., :D].contiguous()
        if Q.stride(-1) != 1 or Q.stride(-2) != D:
            Q = Q.contiguous()
        if K.stride(-1) != 1 or K.stride(-2) != D:
            K = K.contiguous()
        if (V.stride(-1) != 1 or V.stride(-2) != D
                or V.stride(0) != K.stride(0) or V.stride(1) != K.stride(1)):
            V = V.contiguous()
            K = K.contiguous()
        return _hip_ops.attn_fwd(Q, K, V,
                                 mask.contiguous() if mask is not None else None,
                                 causal, scale)
    return torch_ref.attn_fwd(Q, K, V, mask, causal, scale)


def ivf_score(slabs, lens, probes, q):
    """Batched IVF chunk scoring: slabs [nchunks, cap, H] f32, lens
    [nchunks] i32, probes [Q, nprobe] i32, q [Q, H] f32 ->
    [Q, nprobe, cap] f32 (-inf at pad rows)."""
    _require_hip()
    return _hip_ops.ivf_score(slabs, lens, probes, q.contiguous())


def varlen_block_map(cu_seqlens: torch.Tensor, qblk: int = 128):
    """Host-built (seq, qblock) map for attn_varlen: one entry per
    128-row q block of each sequence. cu_seqlens int32 [B+1] (either
    device). Returns (blk_seq, blk_qb) int32 on cu's device."""
    cu = cu_seqlens.to("cpu", torch.int64)
    lens = cu[1:] - cu[:-1]
    nqb = torch.div(lens + qblk - 1, qblk, rounding_mode="floor")
    total = int(nqb.sum())
    blk_seq = torch.repeat_interleave(
        torch.arange(len(lens), dtype=torch.int64), nqb
    )
    # vectorized within-sequence block index: position minus the
    # sequence's first position
    starts = torch.zeros(len(lens), dtype=torch.int64)
    if len(lens) > 1:
        starts[1:] = nqb.cumsum(0)[:-1]
    blk_qb = (torch.arange(total, dtype=torch.int64)
              - torch.repeat_interleave(starts, nqb))
    dev = cu_seqlens.device
    return blk_seq.int().to(dev), blk_qb.int().to(dev)


def attn_varlen(Q, K, V, cu_seqlens, block_map=None, scale=None):
    """Varlen (packed, cu_seqlens) bidirectional attention.
    Q/K/V [total_tokens, H(KV), D]; returns [total_tokens, H, D].
    The protein-path replacement for faesm's flash-attn varlen
    (reference distllm/embed/encoders/esm2.py:41-55)."""
    D = Q.shape[-1]
    if scale is None:
        scale = 1.0 / math.sqrt(D)
    if Q.is_cuda:
        _require_hip()
        if block_map is None:
            block_map = varlen_block_map(cu_seqlens)
        blk_seq, blk_qb = block_map
        if D not in (64, 128):
            Dp = 64 if D < 64 else 128
            pad = Dp - D
            O = _hip_ops.attn_varlen(
                torch.nn.functional.pad(Q, (0, pad)).contiguous(),
                torch.nn.functional.pad(K, (0, pad)).contiguous(),
                torch.nn.functional.pad(V, (0, pad)).contiguous(),
                cu_seqlens.int(), blk_seq, blk_qb, scale)
            return O[..., :D].contiguous()
        if not all(t.stride(2) == 1 and t.stride(1) == D
                   and t.stride(0) == s and s % 8 == 0
                   and t.data_ptr() % 16 == 0
                   for t, s in ((Q, Q.stride(0)), (K, K.stride(0)),
                                (V, K.stride(0)))):
            Q, K, V = (t.clone(memory_format=torch.contiguous_format)
                       for t in (Q, K, V))
        return _hip_ops.attn_varlen(Q, K, V, cu_seqlens.int(), blk_seq,
                                    blk_qb, scale)
    return torch_ref.attn_varlen(Q, K, V, cu_seqlens, scale)


def rope_apply(x, cs, sn, pos, rope_heads: int = -1):
    """Heads >= rope_heads (when >= 0) pass through unchanged — lets a
    fused qkv tensor rope its q|k heads and copy v in ONE launch."""
    if x.is_cuda:
        _require_hip()
        return _hip_ops.rope_apply(x.contiguous(), cs, sn, pos.int(),
                                   rope_heads)
    return torch_ref.rope_apply(x, cs, sn, pos, rope_heads)


def rope_qk_(x, cs, sn, pos, heads: int):
    """Rotates the first `heads` heads of every row of x [..., Hx, D] in
    place (queries and keys of a fresh projection; values stay) and returns
    x."""
    if x.is_cuda and x.shape[-1] in (64, 128) and x.is_contiguous() \
            and x.data_ptr() % 16 == 0:
        _require_hip()
        _hip_ops.rope_inplace(x, cs, sn, pos.int().contiguous(), heads)
        return x
    return x.copy_(rope_apply(x, cs, sn, pos, rope_heads=heads))


def _turns(qkv, pos):
    """Whether attention rotates the queries of qkv as it reads them."""
    return (qkv.is_cuda and qkv.shape[-1] in (64, 128)
            and qkv.dtype == torch.bfloat16 and qkv.is_contiguous()
            and qkv.data_ptr() % 16 == 0 and not _recorded(qkv, pos))


def rope_attn_(qkv, cs, sn, pos, H, HKV, mask=None, causal=False, scale=None):
    """Attention of a fresh projection qkv [B, S, H + 2 HKV, D], whose queries and
    keys are first rotated by the angles of pos [B * S]: the keys in place, the
    queries, which nothing else reads, on their way into attention. Not of rows
    shorter than a quarter of a head: a workgroup has 128 queries of a row, and waits
    for the angles of a few as long as for all of theirs. Rotation and attention in a
    graph, own time over that of two launches, 400 to 16384 tokens: 32 heads of 128 on
    8, rows of 8 1.0 to 1.17, of 16 0.95 to 1.11, of 32 0.88 to 1.03, of 60 0.89 to
    1.01, of 128 0.86 to 1.01, of 1024 0.92 to 0.96; 20 heads of 64, rows of 8 0.94
    to 1.04, of 16 0.90 to 0.99, longer 0.85 to 1.03."""
    k, v = qkv[:, :, H: H + HKV], qkv[:, :, H + HKV:]
    if not _turns(qkv, pos) or qkv.shape[1] < qkv.shape[-1] // 4:
        qkv = rope_qk_(qkv, cs, sn, pos, H + HKV)
        return attn_fwd(qkv[:, :, :H], k, v, mask=mask, causal=causal,
                        scale=scale)
    _require_hip()
    pos = pos.int().contiguous()
    _hip_ops.rope_inplace(qkv, cs, sn, pos, HKV, H)
    return _hip_ops.attn_fwd(
        qkv[:, :, :H], k, v, mask.contiguous() if mask is not None else None,
        causal, scale if scale is not None else 1.0 / math.sqrt(qkv.shape[-1]),
        cs, sn, pos)


def rope_attn_varlen_(qkv, cs, sn, pos, H, HKV, cu_seqlens, block_map=None,
                      scale=None):
    """rope_attn_ of packed rows qkv [T, H + 2 HKV, D] (attn_varlen)."""
    k, v = qkv[:, H: H + HKV], qkv[:, H + HKV:]
    if not _turns(qkv, pos):
        qkv = rope_qk_(qkv, cs, sn, pos, H + HKV)
        return attn_varlen(qkv[:, :H], k, v, cu_seqlens, block_map, scale)
    _require_hip()
    pos = pos.int().contiguous()
    _hip_ops.rope_inplace(qkv, cs, sn, pos, HKV, H)
    if block_map is None:
        block_map = varlen_block_map(cu_seqlens)
    return _hip_ops.attn_varlen(
        qkv[:, :H], k, v, cu_seqlens.int(), *block_map,
        scale if scale is not None else 1.0 / math.sqrt(qkv.shape[-1]),
        cs, sn, pos)


def _embeds(word, pos, type_row):
    return (word.is_cuda and word.dtype == torch.bfloat16
            and word.shape[1] % 8 == 0
            and all(t.is_contiguous() for t in (word, pos, type_row)))


def embed_layer_norm(ids, pos_ids, word, pos, type_row, w, b, eps):
    """Layer norm of word[ids] + pos[pos_ids] + type_row; pos_ids None:
    positions 0, 1, ... of every row of ids [B, S]."""
    if _embeds(word, pos, type_row):
        _require_hip()
        return _hip_ops.embed_layer_norm(
            ids.contiguous(), None if pos_ids is None
            else pos_ids.contiguous(), word, pos, type_row, w, b, eps)
    p = pos[: ids.shape[1]][None] if pos_ids is None else pos[pos_ids]
    return layer_norm(word[ids] + p + type_row, w, b, eps=eps)


def embed_with_bias(ids, pos_ids, mask, word, pos, type_row, w, b, eps):
    """embed_layer_norm, and key_bias of mask: in one launch where both are the
    kernels' and mask has a number per token, unless one of them has been replaced
    and is to see its own."""
    if (embed_layer_norm is _EMBED and key_bias is _KEY_BIAS
            and _embeds(word, pos, type_row) and mask.shape == ids.shape
            and mask.device == ids.device and not mask.is_floating_point()
            and not mask.is_complex() and mask.element_size() in (1, 4, 8)):
        _require_hip()
        return _hip_ops.embed_with_bias(
            ids.contiguous(), None if pos_ids is None
            else pos_ids.contiguous(), word, pos, type_row, w, b, eps,
            mask.contiguous())
    return (embed_layer_norm(ids, pos_ids, word, pos, type_row, w, b, eps),
            key_bias(mask))


def key_bias(mask):
    """Additive key mask of the attention: 0 where mask is not zero, -inf
    where it is."""
    if mask.is_cuda and not mask.is_floating_point() \
            and mask.element_size() in (1, 4, 8):
        _require_hip()
        return _hip_ops.key_bias(mask.contiguous())
    return torch.where(
        mask.bool(),
        torch.zeros((), device=mask.device, dtype=torch.float32),
        torch.full((), float("-inf"), device=mask.device,
                   dtype=torch.float32),
    )


_EMBED, _KEY_BIAS = embed_layer_norm, key_bias


def bert_few_rows(x, mask_f, layers, heads, eps, act):
    """All layers (post-normed, each a tuple of its twelve tensors, see
    csrc/encoder_layers.cpp) of a BERT-class encoder on x [B, S, H] in one
    call; None where rows, types, layouts or sizes (one layer's or another's)
    want the general path, layer by layer: the rules are those of linear's
    products of few rows, with which every product here would be made, and of
    the attention's native head sizes."""
    M, H = x.shape[0] * x.shape[1], x.shape[2]
    if not (x.is_cuda and x.dtype == torch.bfloat16 and 0 < M <= 64
            and act in (ACT_GELU_TANH, ACT_GELU_ERF)
            and H // heads in (64, 128) and H % heads == 0
            and "DISTLLM_GEMM" not in os.environ):
        return None
    w1, w2 = layers[0][6], layers[0][8]
    for w in (layers[0][0], w1, w2):
        if w.shape[0] % 64 or w.shape[1] % 64 or w.shape[1] < 128:
            return None
    _require_hip()
    return _hip_ops.bert_few_rows(x.contiguous(), mask_f,
                                  [t for p in layers for t in p], heads, eps,
                                  _DECODE_ACT[act])


def gateup_swiglu(x, wgup, bias=None):
    """silu(x @ Wg^T) * (x @ Wu^T) with Wg|Wu packed as wgup [2I, K].
    Few rows, and many where _wide_tile says so: ONE product with the swiglu in
    the same launch; otherwise one big GEMM + packed swiglu."""
    orig_shape = x.shape
    x2 = x.reshape(-1, orig_shape[-1])
    M, K = x2.shape
    I = wgup.shape[0] // 2
    if x.is_cuda:
        _require_hip("_hip_gemm")
        if _few_rows(x2, wgup, bias, 128):
            out = _hip_ops.decode_gemm(x2, wgup, bias, 0, 1)
            return out.reshape(*orig_shape[:-1], I)
        tile = _wide_tile(x2, wgup, bias, _WIDE_SWIGLU)
        if tile:
            return _hip_ops.wide_gemm(x2, wgup, bias, _WIDE_SWIGLU,
                                      tile).view(*orig_shape[:-1], I)
    gu = linear(x2, wgup, bias)
    if gu.is_cuda:
        out = _hip_ops.swiglu_packed(gu.contiguous())
    else:
        out = swiglu(gu[:, :I], gu[:, I:])
    return out.reshape(*orig_shape[:-1], I)


def gateup_clamped_glu(x, wgup, limit, alpha, shift):
    """Clamped gated unit of x @ Wg^T and x @ Wu^T, Wg|Wu packed as wgup
    [2I, K]: min(g, limit) * sigmoid(alpha * g) * (clamp(u) + shift), all
    with the clamped g. ONE launch where gateup_swiglu has one."""
    if x.is_cuda:
        _require_hip("_hip_gemm")
        if _few_rows(x, wgup, None, 128):
            return _hip_ops.decode_gemm(x, wgup, None, 0, 2, limit, alpha,
                                        shift)
        tile = _wide_tile(x, wgup, None, _WIDE_CLAMPED)
        if tile:
            return _hip_ops.wide_gemm(x, wgup, None, _WIDE_CLAMPED, tile,
                                      limit, alpha, shift)
        return _hip_ops.clamped_glu(linear(x, wgup), limit, alpha, shift)
    return torch_ref.clamped_glu(linear(x, wgup), limit, alpha, shift)


def quantize_fp8_rows(w: torch.Tensor):
    """Per-output-channel OCP fp8-e4m3 weight quantization for the
    W8A16 decode GEMV: returns (wq uint8 [N, K], scale f32 [N]) with
    scale = absmax/448 so dequant is wq * scale per row."""
    wf = w.detach().float()
    scale = (wf.abs().amax(1) / 448.0).clamp_min(1e-12)
    q = (wf / scale[:, None]).clamp(-448.0, 448.0)
    q = q.to(torch.float8_e4m3fn).view(torch.uint8)
    return q.contiguous(), scale.contiguous()


def gemv_fp8(x, wq, scale, bias=None):
    """out = x @ (dequant(wq) * scale)^T (+bias). x bf16 [M<=8, K],
    wq uint8 fp8-e4m3 [N, K], scale f32 [N]. The fp32 dot runs on the
    quantized values, the channel scale applies after — see
    csrc/gemv_fp8.hip."""
    _require_hip()
    return _hip_ops.gemv_fp8(x.contiguous(), wq, scale, bias)


def gateup_swiglu_fp8(x, wq, scale, bias=None):
    """silu(x @ Wg^T) * (x @ Wu^T) with Wg|Wu packed and quantized as for
    gemv_fp8; bias, of both, is added ahead of the unit."""
    _require_hip()
    if wq.shape[1] % 128 == 0:
        return _hip_ops.gemv_fp8(x.contiguous(), wq, scale, bias, True)
    return _hip_ops.swiglu_packed(gemv_fp8(x, wq, scale, bias))


rope_tables = torch_ref.rope_tables


def _score_fills(Q, N, K):
    """Whether the tiles of score.hip (64, 128 or 256 queries by 128 rows, a
    workgroup each) use the card well enough: by rounds of 256 of them, the
    share of the scores among what the rounds could make. Measured against the
    library's product over 33 to 1000 queries, 8000 to 250000 rows, K of 64 to
    4096, own time over its: from 65 queries on a share of 0.55 and more 0.55 to
    1.08, of 0.4 to 0.55 0.55 to 1.4, below up to 1.6; up to 64, where both are
    bound by the rows, of 0.65 and more 0.65 to 1.0, 63 of 20000 x 4096 (0.6)
    1.39, 33 of 16384 x 4096 1.75. Short sums, which the library's launches cost
    more: up to 64 queries at K <= 384 0.45 to 1.0, one tile of queries at K <=
    128 of up to 66000 rows 0.45 to 0.95. Fewer than 128 workgroups were not
    worth it at all."""
    tile = 64 if Q <= 64 else 128 if Q <= 128 else 256
    wgs = -(-Q // tile) * -(-N // 128)
    if wgs < 128:
        return False
    share = Q * N / (-(-wgs // 256) * 256 * tile * 128)
    return (share >= (0.65 if Q <= 64 else 0.55) or (Q <= 64 and K <= 384)
            or (Q <= 256 and K <= 128 and N <= 1 << 16))


def score(q, corpus):
    """q [Q, K] against the rows of corpus [N, K], float32.

    From 33 queries on, and where its tiles fill the card (_score_fills), the
    product of score.hip; else the library's. Measured against 250000 rows of
    768, us, library and own: 32 queries 168, 171; 64 214, 190; 128 399, 293;
    256 722, 489."""
    Q, K = q.shape
    N = corpus.shape[0]
    if (q.is_cuda and q.device == corpus.device and 32 < Q < 1 << 20
            and q.dtype == corpus.dtype == torch.float32
            and K % 32 == 0 and 32 <= K < 1 << 20 and N <= (1 << 31) - 256
            and Q * N < 1 << 39 and _score_fills(Q, N, K)
            and corpus.is_contiguous() and q.is_contiguous()
            and q.data_ptr() % 16 == 0 and corpus.data_ptr() % 16 == 0):
        _require_hip()
        return _hip_ops.score(q, corpus)
    return q @ corpus.t()


def _score_topk_fills(Q, N, K):
    """Whether score_topk's launches are faster than the scores, by the library,
    and topk. By the share of the scores among what the rounds of the card's 256
    CUs could make, own time over theirs, 33 to 513 queries, 4000 to 250000 rows:
    - two f16 parts (score.hip: from 65 queries and K = 256 on) from 0.3 on 0.44
      to 1.01, below, which is tiles of a few thousand rows, up to 1.7; more than
      256 queries of less than 384 columns, whose launches are the most of it, up
      to 4 million scores 0.8 to 1.27, beyond 0.52 to 0.85;
    - three bf16 parts, K <= 384, one tile of queries 0.34 to 1.0, several from
      0.5 on 0.5 to 0.8, below up to 1.1; K <= 1024 from 0.25 on 0.63 to 0.98,
      below up to 1.07; K of 1536 from 0.65 on 0.79 to 0.98, below up to 1.7."""
    tile = 64 if Q <= 64 else 128 if Q <= 128 else 256
    queries, rows = -(-Q // tile), -(-N // 128)
    if Q > 64 and K >= 256:
        each = min(max(256 // queries, 1), rows)
        rounds = -(-queries * each // 256) * -(-rows // each)
        least = 0.3
        if Q > 256 and K < 384 and Q * N < 4_000_000:
            return False
    else:
        rounds = -(-queries * rows // 256)
        least = (0.65 if K > 1024 else 0.25 if K > 384 else
                 0 if Q <= 256 else 0.5)
    return Q * N >= least * rounds * 256 * tile * 128


def _search_few_fills(Q, N, K):
    """Whether one to four queries go by search_few (topk_search.hip): measured
    against the library's product and topk, own time over theirs, k to 30. One
    query, 64 to 1024 columns, from 10000 rows on 0.43 to 0.96, 8192 rows 0.88 to
    1.15, below up to 1.3; two, from 128 columns on, 0.47 to 1.0, of 64 up to 1.1.
    Three and four of 128 to 768 columns to 32768 rows 0.58 to 1.0; beyond, of 384
    0.95 to 1.07, of 128 up to 1.3; of 64 up to 1.6, of more than 768, whose sums
    leave no room for rows, up to 1.5. Of 544, 640 and 768 columns the library's time
    jumps by a factor of two from one size to the next beyond 60000 rows, and own
    time lies between: at 18 sizes from 33000 to 200000 rows 0.45 to 0.97 but for
    120000 and 180000 of 544 and 130000 and 190000 of all, 1.03 to 1.11. Beyond it is
    as it is below (215000 to 300000 rows 0.48 to 0.59 and 1.04 to 1.13, 250000 among
    the latter), and left to the library."""
    if N < 10000 or K % 4 or K < (64 if Q == 1 else 128):
        return False
    return K <= 1024 if Q <= 2 else Q <= 4 and K <= 768 and (
        N <= 32768 or (K > 512 and N <= 200000))


class NarrowRows(NamedTuple):
    """Rows of a corpus in 16 bits beside it (narrow_search.hip). They are its
    until it is written to: holds says whether that was counted, and who keeps
    them sees to it that nothing writes uncounted (through `.data`, by a kernel, by
    a replayed graph), after which they would choose wrong rows."""
    rows: torch.Tensor      # f16 [N, K in whole 64s], of the rows times 2^up
    up: int
    error: float            # most that a row and its 16 bits are apart
    norm: float             # most that those are long, both times 2^up
    corpus: torch.Tensor
    version: int

    def holds(self, corpus) -> bool:
        return self.corpus is corpus and self.version == corpus._version


def narrow_rows(corpus):
    """NarrowRows of a corpus [N, K] on a GPU, for found_narrow; None where they
    would be of no use or there is no room for them: numbers that are infinite
    or NaN, rows whose lengths differ so much that what the longest loses in 16
    bits hides the others, more than an eighth of the memory that is free."""
    if not (corpus.is_cuda and corpus.dtype == torch.float32
            and corpus.dim() == 2 and corpus.is_contiguous()
            and not corpus.is_inference()
            and corpus.shape[0] > 0 and 0 < corpus.shape[1] < 1 << 16
            and corpus.shape[1] % 4 == 0 and corpus.data_ptr() % 16 == 0):
        return None
    held = corpus.shape[0] * max(128, (corpus.shape[1] + 63) // 64 * 64) * 2
    if (not hasattr(_hip_ops, "narrow_rows")
            or held > torch.cuda.mem_get_info(corpus.device)[0] // 8):
        return None
    version = corpus._version
    try:
        made = _hip_ops.narrow_rows(corpus)
    except torch.OutOfMemoryError:
        return None
    if made is None:
        return None
    rows, up, error, norm, usual = made
    # sums of squares in float32 are a little off
    return (NarrowRows(rows, up, error * 1.0001, norm * 1.0001, corpus,
                       version) if norm <= 4 * usual else None)


def _narrow_fills(Q, N, K, k):
    """Whether found_narrow is faster than score_topk of queries copied to the
    GPU and found_lists of that: half of the rows' bytes are spared, and the rows
    that may be among the best, more with k, are read by one workgroup of each
    query. Unit vectors, own time over theirs:
    - to 1536 columns, 64 to 250000 rows, up to 256 queries 0.32 to 1.00, but
      for 17 and more queries of few thousand rows and large k, 0.95 to 1.13
      (1536 columns, 4000 rows, k = 60, one query 1.04); 600 and 1000 queries
      from 2048 rows on 0.37 to 1.0 (of 2000 to 4000 and large k up to 1.10),
      of fewer 0.98 to 1.08;
    - beyond by k and the rows. 2048 columns, k of 1, 10, 60, the slowest of 1
      to 256 queries: 1000 rows 1.01, 1.05, 1.40, 4000 0.91, 0.97, 1.52, 32000
      0.70, 0.77, 0.94; 4096: 4000 rows 1.37, 1.47, 2.28, 16000 0.89, 0.99,
      1.55, 32000 0.72, 0.78, 1.31, 125000 0.60, 0.64, 0.97; 8192: 4000 rows
      1.8, 2.1, 3.8, 32000 0.72, 1.03, 2.2, 125000 0.60, 0.70, 1.20; 16384,
      64000 rows 0.91, 1.43, above 2. 600 and 1000 queries of 4096: 4000 rows
      0.95, 0.98, 1.21, 16000 0.81, 0.89, 1.04; 8192: 16000 0.75, 0.91, 1.19,
      64000 0.49, 0.57, 0.93."""
    if K > 8192 or (Q > 256 and N < 2048):
        return False
    if K > 1536:
        return N >= K * (1 + 0.12 * k if Q > 256 else 2.6 + 0.4 * k)
    return K * k <= 26000 or N >= 8000 or (Q <= 16 and K * k <= 80000)


def found_narrow(q, corpus, k, narrow, general=None):
    """found_lists of score_topk for queries [Q, K] of the host, by way of the
    corpus's NarrowRows: None where that is not the faster way, or there is no room
    for what it takes. Queries that these cannot answer (infinite or NaN numbers,
    of far more rows nearly as good as the best) go on to general(queries, k),
    on the corpus's device, score_topk of them if it is not given."""
    Q, K = q.shape
    N = corpus.shape[0]
    if not (0 < Q < 1 << 20 and 0 < k <= min(60, N)
            and q.dtype == torch.float32 and q.device.type == "cpu"
            and tuple(corpus.shape[1:]) == (K,) and narrow.holds(corpus)
            and _narrow_fills(Q, N, K, k) and q.is_contiguous()
            and 0 < _hip_ops.narrow_bytes(Q, N, K, narrow.rows.shape[1])
            <= 1 << 31):
        return None
    try:
        found = _hip_ops.narrow_found(q, corpus, narrow.rows, narrow.up,
                                      narrow.error, narrow.norm, k, True)
    except torch.OutOfMemoryError:
        return None
    scores, indices, rest = found
    if rest:
        left = (q if len(rest) == Q else q[rest]).to(corpus.device)
        v, i = (general(left, k) if general is not None
                else score_topk(left, corpus, k))
        for at, s, x in zip(rest, *found_lists(v.float(), i.int())):
            scores[at], indices[at] = s, x
    return scores, indices


def score_topk(q, corpus, k):
    """The k best rows of corpus [N, K] for every q [Q, K], as topk of score has
    them: (values [Q, k], indices [Q, k] int32).

    A few queries, where _search_few_fills, are multiplied in float32 by the kernel
    that also chooses their rows.
    For 33 and more queries and k to 60 without the matrix of scores, where
    _score_topk_fills: the largest score of every four rows, the k best of these
    fours, and their rows once more in float32. 250000 rows of 768, k = 10, us,
    with the matrix and without: 64 queries 211, 202; 128 333, 228; 256 565, 333
    (517 to 840 where f16 parts do not do, see score.hip)."""
    Q, K = q.shape
    N = corpus.shape[0]
    if (0 < Q <= 4 and 0 < k <= min(30, N) and q.is_cuda
            and q.device == corpus.device
            and q.dtype == corpus.dtype == torch.float32
            and tuple(corpus.shape[1:]) == (K,)
            and N < (1 << 31) - 256 and _search_few_fills(Q, N, K)
            and corpus.is_contiguous() and q.is_contiguous()
            and q.data_ptr() % 16 == 0 and corpus.data_ptr() % 16 == 0):
        _require_hip()
        return _hip_ops.search_few(q, corpus, k)
    if (32 < Q < 1 << 20 and 0 < k <= min(60, N)
            and q.is_cuda and q.device == corpus.device
            and q.dtype == corpus.dtype == torch.float32
            and K % 32 == 0 and 32 <= K < 1 << 20 and N <= (1 << 31) - 256
            and Q * N < 1 << 39 and _score_topk_fills(Q, N, K)
            and corpus.is_contiguous() and q.is_contiguous()
            and q.data_ptr() % 16 == 0 and corpus.data_ptr() % 16 == 0):
        _require_hip()
        return _hip_ops.score_topk(q, corpus, k)
    return topk(score(q, corpus).contiguous(), k)


def _topk_in_registers(Q, N, k):
    """Whether workgroups hold their chunks in registers (topk_regs_kernel).
    Measured, both rounds, against the radix select: k up to 60 0.2 to 0.9 of
    its time everywhere (1 to 5000 rows of 300 to 4 million); k = 65, 100, 128
    from 4096 scores on 0.3 to 0.9, 2048 rows of 1000 1.4, 1.4, 1.2, 64 rows of
    1000 0.7; k = 200 of 1 to 512 rows 0.4 to 1.0, of 2048 rows 0.9 to 1.6;
    k = 255 1.3 to 4."""
    return 0 < k <= 60 or (k <= 128 and N >= 4000) or (k <= 200 and Q <= 512)


def topk(scores, k, chunk=1 << 15):
    """Row-wise top-k over a [Q, N] f32 score matrix.

    GPU: chunks of scores by workgroups, then rounds over the candidates.
    Chunks of 8192 in registers for small k (_topk_in_registers); else a radix
    select reads chunks of `chunk` (the 32k default keeps the grid >= 1024
    workgroups even for a few queries).
    Returns (values [Q,k] f32 desc-sorted, indices [Q,k] int32).
    """
    if scores.is_cuda:
        _require_hip()
        Q, N = scores.shape
        k_eff = min(k, N)
        few = k_eff > 0 and _topk_in_registers(Q, N, k_eff)
        if few:
            chunk = min(chunk, 8192)
        v, i = _hip_ops.topk_chunked(scores.contiguous(), None, k_eff, chunk,
                                     few)
        while v.shape[1] > k_eff:  # candidates of several chunks
            v, i = _hip_ops.topk_chunked(
                v, i, k_eff, 8192 if few else v.shape[1], few)
        if k_eff < k:
            pad_v = torch.full((Q, k - k_eff), float("-inf"),
                               device=v.device)
            pad_i = torch.full((Q, k - k_eff), -1, dtype=torch.int32,
                               device=v.device)
            v = torch.cat([v, pad_v], 1)
            i = torch.cat([i, pad_i], 1)
        return v[:, :k], i[:, :k]
    return torch_ref.topk(scores, min(k, scores.shape[1]))


def found_lists(v, i):
    """Scores and indices [Q, k] on a GPU (float32, int32) as lists of their
    rows, without the entries whose index is negative."""
    _require_hip()
    return _hip_ops.found_lists(v, i)


def hamming_score(qcodes, codes_t):
    if qcodes.is_cuda:
        _require_hip()
        return _hip_ops.hamming_score(qcodes.contiguous(),
                                      codes_t.contiguous())
    return torch_ref.hamming_score(qcodes, codes_t)


def sample_tokens(logits, rand, temp, min_p=0.0):
    if logits.is_cuda:
        _require_hip()
        return _hip_ops.sample_tokens(logits.float().contiguous(),
                                      rand.float(), temp, min_p)
    return torch_ref.sample_tokens(logits, rand, temp, min_p)


def paged_attn(q, kcache, vcache, block_table, ctx_len, scale=None):
    if scale is None:
        scale = 1.0 / math.sqrt(q.shape[-1])
    if q.is_cuda:
        _require_hip()
        return _hip_ops.paged_attn(q.contiguous(), kcache, vcache,
                                   block_table.int(), ctx_len.int(), scale)
    return torch_ref.paged_attn(q, kcache, vcache, block_table, ctx_len,
                                scale)


def cache_put(knew, vnew, kcache, vcache, block_table, slot):
    if knew.is_cuda:
        _require_hip()
        _hip_ops.cache_put(knew.contiguous(), vnew.contiguous(), kcache,
                           vcache, block_table.int(), slot.int())
        return
    # CPU reference: scatter
    B, HKV, D = knew.shape
    BLK = kcache.shape[2]
    for b in range(B):
        pos = int(slot[b])
        blk = int(block_table[b, pos // BLK])
        kcache[blk, :, pos % BLK] = knew[b]
        vcache[blk, :, pos % BLK] = vnew[b]


def rope_put(qkv, cs, sn, ctx, kcache, vcache, block_table, bias=None):
    """A decode step's projections [B, H + 2 HKV, D]: queries and keys are
    rotated by position ctx - 1; queries are returned [B, H, D], keys and
    values go to that position of the cache, in one launch. qkv may be the
    fp32 slabs [S, B, H + 2 HKV, D] of linear_parts (heads of 64 and 128),
    with the bias that they lack."""
    if qkv.is_cuda and qkv.shape[-1] in (64, 128):
        _require_hip()
        return _hip_ops.rope_put(qkv.contiguous(), cs, sn, ctx.int(), kcache,
                                 vcache, block_table.int(),
                                 bias if qkv.dim() == 4 else None)
    H = qkv.shape[1] - 2 * kcache.shape[1]
    slot = (ctx - 1).int()
    qkv = rope_apply(qkv, cs, sn, slot, rope_heads=H + kcache.shape[1])
    cache_put(qkv[:, H: H + kcache.shape[1]].contiguous(),
              qkv[:, H + kcache.shape[1]:].contiguous(), kcache, vcache,
              block_table, slot)
    return qkv[:, :H].contiguous()


def step_plan(layers, ctx, H, kcache, block_table):
    """What step_attn of so many layers needs, an item for each: the shares of
    the sequences, cut by their lengths, and its counters. None for heads and
    devices that need nothing."""
    HKV, D = kcache.shape[1], kcache.shape[3]
    if not kcache.is_cuda or D not in (64, 128):
        return [None] * layers
    _require_hip()
    slots, zeros = _hip_ops.step_plan(ctx.int(), block_table.int(), layers, H,
                                      HKV, kcache.dtype == torch.uint8)
    return [(slots, row) for row in zeros.unbind()]


def step_begin(tokens, emb, w_norm, eps, layers, ctx, H, kcache, block_table):
    """The rows x [B, 1, n] of tokens [B] in the table emb, the RMS norm of x times
    w_norm, and step_plan of the others: where the step has a plan, the norm in its
    launch. (The rows are torch's to take, which refuses a token outside the table; a
    launch that took them too was 3 to 6 us less.) With this and the head's product by
    norm_linear(..., f32=True) a step of eight layers of 4096 takes, us, one row of
    2048 tokens 792 -> 786, with 8-bit weights 583 -> 577, 64 rows 1476 -> 1457."""
    x = emb[tokens.long()].unsqueeze(1)
    if (layers > 0 and kcache.is_cuda and kcache.shape[3] in (64, 128)
            and x.device == w_norm.device == kcache.device
            and x.dim() == 3 and 0 < x.shape[2] <= 8192
            and x.shape[2] % 8 == 0 and w_norm.shape == x.shape[2:]
            and all(t.dtype == torch.bfloat16 and t.is_contiguous()
                    and t.data_ptr() % 16 == 0 for t in (x, w_norm))
            and not _recorded(x, w_norm)):
        _require_hip()
        slots, zeros, h = _hip_ops.step_plan(
            ctx.int(), block_table.int(), layers, H, kcache.shape[1],
            kcache.dtype == torch.uint8, x, w_norm, eps)
        return x, h, [(slots, row) for row in zeros.unbind()]
    return (x, rms_norm(x, w_norm, eps=eps),
            step_plan(layers, ctx, H, kcache, block_table))


def step_inputs(to, tokens, lengths, slots, blocks):
    """What a captured decode step reads, from lists into tensors of the host, to:
    tokens [B] int64, lengths [B], slots [B or 0], block table [B, width], int32.
    Rows past those of the lists have length 1, token, slot and blocks 0. (A row's
    blocks as tensors of their own took 32 sequences 100 us.)"""
    _hip_ops.step_inputs(*to, tokens, lengths, slots, blocks)


def step_attn(qkv, cs, sn, ctx, kcache, vcache, block_table, bias, scale,
              plan, ahead=None):
    """rope_put and the attention of its queries over the cache, the new tokens
    of all rows among it (of a sequence several rows may be one token each, in
    any order) -> [B, H, D]; one launch for heads of 64 and 128. plan: an item of
    step_plan, used up. ahead: weights of the product that follows, which few
    sequences leave the time to fetch into the caches."""
    if qkv.is_cuda and qkv.shape[-1] in (64, 128):
        _require_hip()
        return _hip_ops.step_attn(qkv.contiguous(), cs, sn, ctx.int(), kcache,
                                  vcache, block_table.int(),
                                  bias if qkv.dim() == 4 else None, scale,
                                  *plan, ahead)
    q = rope_put(qkv, cs, sn, ctx, kcache, vcache, block_table, bias)
    return paged_attn(q, kcache, vcache, block_table, ctx, scale)


# ---- sandwich-norm / latent-attention decoder -----------------------------

def embed_norm(tokens, table, w_next, n, eps):
    """Start of the residual stream: x = table[token] in fp32 and h =
    rms(x) * w_next, statistics over the first n columns. -> (h, x)"""
    if table.is_cuda:
        _require_hip("_hip_residual")
        x = torch.empty(tokens.shape[0], table.shape[1],
                        dtype=torch.float32, device=table.device)
        h = _hip_ops.sandwich_norm(table, tokens, x, None, w_next, n, eps)
        return h, x
    return torch_ref.embed_norm(tokens, table, w_next, n, eps)


def post_norm_add(y, x, w_post, w_next, n, eps):
    """End of a sandwich-normed sublayer: x += rms(y) * w_post (x fp32,
    in place), returns the next sublayer's input rms(x) * w_next. y may be
    what linear_parts returned."""
    if y.is_cuda:
        _require_hip("_hip_residual")
        return _hip_ops.sandwich_norm(y, None, x, w_post, w_next, n, eps)
    return torch_ref.post_norm_add(y, x, w_post, w_next, n, eps)


def latent_prep(ab, q_cols, q_rank, rank, wq, wc, eps, cache, block_table,
                row_seq, ctx):
    """Norm both down-projections of a latent-attention layer, ab [M, columns]
    or what linear_parts returned, in one launch: the query latent (first
    q_cols columns of ab) is returned, the key/value latent goes straight to
    its cache slot (position ctx - 1 of block-table row row_seq; ctx 0 writes
    nothing). cache None: the layer has no latent of its own."""
    if ab.is_cuda:
        _require_hip("_hip_latent")
        return _hip_ops.latent_prep(ab, q_cols, q_rank, rank, wq, wc, eps,
                                    cache, block_table, row_seq, ctx)
    return torch_ref.latent_prep(ab, q_cols, q_rank, rank, wq, wc, eps,
                                 cache, block_table, row_seq, ctx)


def rotary_latent_prep(ab, heads, dp, tp, rank, wc, eps, table, cache,
                       block_table, row_seq, ctx, ql):
    """What precedes latent attention with rotated parts, on a projection
    ab [M, heads * (dp unrotated, tp rotated numbers) | latent | key part |
    ...], in one launch: the rotated numbers of the queries of the first
    len(ql) rows go to the last tp columns of ql [n, heads, latent + tp],
    those of the others back to ab; normed latents (statistics over rank
    numbers) and rotated key parts go to their cache rows (position ctx - 1;
    ctx 0 writes nothing). cache None: the layer has none of its own."""
    if ab.is_cuda:
        _require_hip("_hip_latent")
        _hip_ops.rotary_latent_prep(ab, heads, dp, tp, rank, wc, eps, table,
                                    cache, block_table, row_seq, ctx, ql)
        return
    torch_ref.rotary_latent_prep(ab, heads, dp, tp, rank, wc, eps, table,
                                 cache, block_table, row_seq, ctx, ql)


def latent_gather(cache, block_table, key_seq, key_pos, rank=None):
    """Cached latents of (sequence, position) pairs, packed. With rank
    (fewer columns than a cache row has): the first rank columns and the
    others, as two tensors."""
    if cache.is_cuda:
        _require_hip("_hip_latent")
        c, rest = _hip_ops.latent_gather(cache, block_table, key_seq,
                                         key_pos, rank or cache.shape[2])
        return c if rank is None else (c, rest)
    c = torch_ref.latent_gather(cache, block_table, key_seq, key_pos)
    return c if rank is None else (c[:, :rank].contiguous(),
                                   c[:, rank:].contiguous())


def head_gemm(x, w, out=None):
    """One product per head: x [M, H, K], w [H, N, K] -> [M, H, N]. Rows
    and heads of x and out may be strided."""
    if x.is_cuda and x.dtype == torch.bfloat16:
        _require_hip("_hip_latent")
        if out is None:
            out = x.new_empty(x.shape[0], x.shape[1], w.shape[1])
        _hip_ops.head_gemm(x, w, out)
        return out
    if x.is_cuda:  # true 32-bit product
        res = torch.bmm(x.transpose(0, 1), w.transpose(1, 2))
        res = res.transpose(0, 1).contiguous()
    else:
        res = torch_ref.head_gemm(x, w)
    if out is None:
        return res
    return out.copy_(res)


def latent_attn(q, cache, block_table, row_seq, ctx, window, scale,
                nsplit=0, rank=None, sink=None, gate=None):
    """Attention of single-token rows over paged latents, queries folded
    into the latent space: q [M, H, R] -> [M, H, R]. A row sees the last
    `window` positions of its sequence up to its own (ctx - 1). nsplit:
    workgroups that share a row's keys (0: chosen from the sizes). With
    rank, only the first rank columns of a cache row are the value. sink
    [H]: exp(sink) is part of the softmax's denominator; gate [M, H]: head
    outputs are multiplied by its sigmoid."""
    rank = rank or cache.shape[2]
    if q.is_cuda:
        _require_hip("_hip_latent")
        return _hip_ops.latent_attn(q, cache, block_table, row_seq, ctx,
                                    window, scale, nsplit, rank, sink, gate)
    return torch_ref.latent_attn(q, cache, block_table, row_seq, ctx,
                                 window, scale, rank, sink, gate)


def latent_attn_values(q, cache, block_table, row_seq, ctx, window, scale, uv,
                       out, nsplit=0, rank=None, sink=None, gate=None):
    """head_gemm of latent_attn's result and uv [H, N, R], to out [M, H, N]: where a
    row's keys are shared, in the launch that joins the shares."""
    if q.is_cuda and q.dtype == torch.bfloat16:
        _require_hip("_hip_latent")
        _hip_ops.latent_attn_values(q, cache, block_table, row_seq, ctx,
                                    window, scale, nsplit,
                                    rank or cache.shape[2], sink, gate, uv,
                                    out)
        return out
    return head_gemm(latent_attn(q, cache, block_table, row_seq, ctx, window,
                                 scale, nsplit, rank, sink, gate), uv, out=out)


def attn_window(q, kv, out, cu_q, cu_k, block_map, window, scale, kr=None,
                sink=None, gate=None):
    """Sliding-window causal attention of packed queries that are the
    last ones of their packed keys (a prompt portion after its cached
    part). q [Tq, H, DK], kv [Tk, H*DK + H*DV], out [Tq, H, DV]. With kr
    [Tk, DR], key numbers that all heads share, queries have DK + DR
    numbers. sink, gate: as for latent_attn."""
    if q.is_cuda:
        _require_hip("_hip_latent")
        blk_seq, blk_qb = block_map
        _hip_ops.attn_window(q, kv, out, cu_q, cu_k, blk_seq, blk_qb,
                             window, scale, kr, sink, gate)
        return out
    return out.copy_(torch_ref.attn_window(q, kv, out.shape[2], cu_q, cu_k,
                                           window, scale, kr, sink, gate))


# ---- chunked attention / delta rule / experts decoder -----------------------

def embed_positions(tokens, ctx, table, pos):
    """Start of a residual stream with position vectors: x = table[token]
    + pos[ctx - 1] in fp32. -> (x in the table's dtype, x)"""
    if table.is_cuda:
        _require_hip("_hip_residual")
        x = torch.empty(tokens.shape[0], table.shape[1],
                        dtype=torch.float32, device=table.device)
        return _hip_ops.embed_positions(tokens, ctx, table, pos, x), x
    return torch_ref.embed_positions(tokens, ctx, table, pos)


def layer_norm_add(y, x, w, b, n, eps, final=None, mix=None):
    """End of a sublayer whose output is layer-normed: x += norm(y) (x
    fp32, in place; statistics over n columns). Returns x in y's dtype,
    normed by final = (weight, bias) if given. With mix [M, top] the
    sublayer output is sum_k mix[m, k] * y[m * top + k]."""
    if y.is_cuda:
        _require_hip("_hip_residual")
        wf, bf = final if final is not None else (None, None)
        return _hip_ops.layer_norm_add(y, x, w, b, n, eps, wf, bf, mix)
    return torch_ref.layer_norm_add(y, x, w, b, n, eps, final, mix)


def attn_prep(ab, heads, kv_heads, dp, vp, dim, wq, wk, eps, pages,
              block_table, row_seq, ctx):
    """Norm the query heads of a fused projection (returned, [M, heads,
    dp]) and its key heads, and write keys and values to their pages
    (position ctx - 1; ctx 0 writes nothing). pages None: the layer has
    no keys and values of its own."""
    if ab.is_cuda:
        _require_hip("_hip_hybrid")
        kp, vpg = pages if pages is not None else (None, None)
        return _hip_ops.attn_prep(ab, heads, kv_heads, dp, vp, dim, wq, wk,
                                  eps, kp, vpg, block_table, row_seq, ctx)
    return torch_ref.attn_prep(ab, heads, kv_heads, dp, vp, dim, wq, wk, eps,
                               pages, block_table, row_seq, ctx)


def paged_attn_rows(q, kpages, vpages, ab, gate_at, out, block_table,
                    row_seq, ctx, chunk, scale, softcap, dist, nsplit=0):
    """Attention of single-token rows over paged keys and values. A row
    sees the positions of its chunk up to its own. The output is gated by
    the sigmoid of ab's columns from gate_at on."""
    if q.is_cuda:
        _require_hip("_hip_chunked")
        _hip_ops.paged_attn_rows(q, kpages, vpages, ab, gate_at, out,
                                 block_table, row_seq, ctx, chunk, scale,
                                 softcap, dist, nsplit)
        return out
    return torch_ref.paged_attn_rows(q, kpages, vpages, ab, gate_at, out,
                                     block_table, row_seq, ctx, chunk, scale,
                                     softcap, dist)


def paged_attn_prompts(q, kpages, vpages, ab, gate_at, out, block_table,
                       prompts, chunk, scale, softcap, dist):
    """The same for the rows of prompt portions (step.PromptBlocks)."""
    if q.is_cuda:
        _require_hip("_hip_chunked")
        _hip_ops.paged_attn_prompts(q, kpages, vpages, ab, gate_at, out,
                                    block_table, prompts.portions,
                                    prompts.blocks, chunk, scale, softcap,
                                    dist)
        return out
    return torch_ref.paged_attn_prompts(q, kpages, vpages, ab, gate_at, out,
                                        block_table, prompts, chunk, scale,
                                        softcap, dist)


def gated_delta(ab, heads, kv_heads, dp, vp, dim, vdim, conv_w, decay,
                o_norm, unit_eps, eps, state, conv, segments, row_seq, ctx):
    """Gated delta rule of a ragged step on the fused projection ab
    [M, queries | keys | values | gates | b | a]: short convolutions, unit
    queries and keys, recurrence in fp32, gated output norm.
    -> [M, heads * vp]; state and convolution slots are updated."""
    if ab.is_cuda:
        _require_hip("_hip_hybrid")
        return _hip_ops.gated_delta(
            ab, heads, kv_heads, dp, vp, dim, vdim, conv_w, decay, o_norm,
            unit_eps, eps, state, conv, segments.row0, segments.rows,
            segments.slot, segments.longest, row_seq, ctx, segments.longs,
            segments.chunks, segments.SHORT)
    return torch_ref.gated_delta(
        ab, heads, kv_heads, dp, vp, dim, vdim, conv_w, decay, o_norm,
        unit_eps, eps, state, conv, segments, row_seq, ctx)


def up_xielu(x, wup, act):
    """xielu(x @ wup^T); act: the activation's two raw numbers."""
    if x.is_cuda:
        _require_hip("_hip_gemm")
        _require_hip("_hip_experts")
        if _few_rows(x, wup):
            return _hip_ops.decode_gemm(x, wup, None, 0, 3, act_nums=act)
        return _hip_ops.xielu(linear(x, wup), act)
    return torch_ref.xielu(linear(x, wup), act)


def route(h, router, ctx, top, groups, keep):
    """Experts of every row: ids [M, top] int32 and their softmax scores.
    Only experts of the `keep` groups with the largest scores count; rows
    with ctx 0 get ids -1 and weights 0."""
    if h.is_cuda:
        _require_hip("_hip_experts")
        if h.dtype == torch.bfloat16 and router.shape[0] <= 256:
            return _hip_ops.route(h, router, ctx, top, groups, keep)
        logits = torch.nn.functional.linear(h.float(), router.float())
        return _hip_ops.route(logits, None, ctx, top, groups, keep)
    return torch_ref.route(h, router, ctx, top, groups, keep)


def experts(h, ids, wup, wdown, gated=True):
    """Experts: row m * top + k of the result is expert ids[m, k] of row m
    (undefined for id -1). Gated units, wup [E, 2F, W]: gate and up rows
    alternate in groups of 16; else squared ReLU, wup [E, F, W]."""
    if h.is_cuda:
        _require_hip("_hip_experts")
        return _hip_ops.experts(h, ids, wup, wdown, gated)
    return torch_ref.experts(h, ids, wup, wdown, gated)


def route_sigmoid(h, router, correction, ctx, top, scale, shards=0):
    """Experts of every row by sigmoid scores: ids [M, top] int32 of the
    largest sums of score and correction, and scale times their scores
    without it. One more row of the router than corrections is the gate of
    an expert that serves every row: its sigmoid is a further column of the
    weights, or, with shards, the weight of that many further choices, the
    experts behind the others. Rows with ctx 0 get ids -1 and weights 0."""
    if h.is_cuda:
        _require_hip("_hip_experts")
        if h.dtype == torch.bfloat16 and router.shape[0] <= 256:
            return _hip_ops.route_sigmoid(h, router, correction, ctx, top,
                                          scale, shards)
        logits = torch.nn.functional.linear(h.float(), router.float())
        return _hip_ops.route_sigmoid(logits, None, correction, ctx, top,
                                      scale, shards)
    return torch_ref.route_sigmoid(h, router, correction, ctx, top, scale,
                                   shards)


def up_relu2(x, wup):
    """The square of relu(x @ wup^T)."""
    if x.is_cuda:
        _require_hip("_hip_gemm")
        if _few_rows(x, wup):
            return _hip_ops.decode_gemm(x, wup, None, 0, 5)
        return _hip_ops.relu2(linear(x, wup))
    return torch_ref.relu2(linear(x, wup))


# ---- parallel attention and delta rule / linear recurrent decoder -----------

def residual_step(x, y=None, bias=None, rms=None, embed=None, vec=None,
                  act=None, fresh=False, dtype=None):
    """One boundary of an fp32 residual stream x [M, W], in place:
      x += y + bias (fp32 vector), or rms(y) * w with rms = (w, n, eps),
           statistics over n columns
      x += scale * table[token] with embed = (tokens, table, scale)
      x += vec (fp32 vector)
    all of them optional; with `fresh` x starts from zeros. Returns x, or
    tanh(alpha x) * w + b with act = (w, b, alpha), in `dtype` (default:
    that of y, of the table without y)."""
    if dtype is None:
        dtype = y.dtype if y is not None else embed[1].dtype
    if x.is_cuda:
        _require_hip("_hip_residual")
        tokens, table, scale = embed if embed is not None else (None, None,
                                                                1.0)
        w_rms, n, eps = rms if rms is not None else (None, x.shape[1], 0.0)
        w, b, alpha = act if act is not None else (None, None, None)
        h = torch.empty(x.shape, dtype=dtype, device=x.device)
        _hip_ops.residual_step(x, y, bias, w_rms, n, eps, tokens, table,
                               scale, vec, w, b, alpha, fresh, h)
        return h
    return torch_ref.residual_step(x, y, bias, rms, embed, vec, act, fresh,
                                   dtype)


def gated_rows(x, wgate, tokens, table, col0, n):
    """gelu_tanh(x @ wgate^T) * table[token, col0: col0 + n], zeros in the
    columns of wgate behind n."""
    if x.is_cuda:
        _require_hip("_hip_gemm")
        if _few_rows(x, wgate):
            return _hip_ops.decode_gemm_rows(x, wgate, 0, tokens, table,
                                             col0, n)
        return _hip_ops.gelu_rows(linear(x, wgate), tokens, table, col0, n)
    return torch_ref.gelu_rows(linear(x, wgate), tokens, table, col0, n)


def rotation_table(ctx, freq, mult):
    """mult * (cos, sin) of freq (fp64) times the position ctx - 1 of every
    row: [M, pairs, 2] fp32."""
    if ctx.is_cuda:
        _require_hip("_hip_residual")
        return _hip_ops.rotation_table(ctx, freq, mult)
    return torch_ref.rotation_table(ctx, freq, mult)


def rotary_prep(ab, heads, kv_heads, dp, dim, wq, wk, eps, table, pages,
                block_table, row_seq, ctx):
    """Norm and rotate the query heads of a projection ab [M, queries |
    keys] (returned, [M, heads, dp]) and its key heads; those go to the key
    pages, keys as projected to the value pages (position ctx - 1; ctx 0
    writes nothing). The first 2 * pairs numbers of a head rotate."""
    if ab.is_cuda:
        _require_hip("_hip_hybrid")
        return _hip_ops.rotary_prep(ab, heads, kv_heads, dp, dim, wq, wk,
                                    eps, table, pages[0], pages[1],
                                    block_table, row_seq, ctx)
    return torch_ref.rotary_prep(ab, heads, kv_heads, dp, dim, wq, wk, eps,
                                 table, pages, block_table, row_seq, ctx)


def sink_attn_rows(q, kpages, vpages, out, block_table, row_seq, ctx, scale,
                   sink, out_scale, nsplit=0):
    """Causal attention of single-token rows over paged keys and values;
    exp(sink) of the head is part of the softmax's denominator. out
    [M, heads * vdim] (rows may be strided) takes the result times
    out_scale."""
    if q.is_cuda:
        _require_hip("_hip_hybrid")
        _hip_ops.sink_attn_rows(q, kpages, vpages, out, block_table, row_seq,
                                ctx, scale, sink, out_scale, nsplit)
        return out
    return torch_ref.sink_attn_rows(q, kpages, vpages, out, block_table,
                                    row_seq, ctx, scale, sink, out_scale)


def sink_attn_prompts(q, kpages, vpages, out, block_table, prompts, scale,
                      sink, out_scale):
    """The same for the rows of prompt portions (step.PromptBlocks)."""
    if q.is_cuda:
        _require_hip("_hip_hybrid")
        _hip_ops.sink_attn_prompts(q, kpages, vpages, out, block_table,
                                   prompts.portions, prompts.blocks, scale,
                                   sink, out_scale)
        return out
    return torch_ref.sink_attn_prompts(q, kpages, vpages, out, block_table,
                                       prompts, scale, sink, out_scale)


def channel_delta(ab, ag, heads, kv_heads, dp, vp, dim, vdim, conv_w, a_log,
                  dt_bias, o_norm, unit_eps, eps, out_scale, state, conv,
                  segments, row_seq, ctx, out):
    """Delta rule with a decay per key channel of a ragged step, on the
    projection ab [M, queries | keys | values | b] and the second product
    ag [M, decays | gates]: short convolutions, unit queries and keys,
    recurrence in fp32, output norm, sigmoid gate, out_scale. out
    [M, heads * vp] (rows may be strided); state and convolution slots are
    updated."""
    if ab.is_cuda:
        _require_hip("_hip_hybrid")
        _hip_ops.channel_delta(
            ab, ag, heads, kv_heads, dp, vp, dim, vdim, conv_w, a_log,
            dt_bias, o_norm, unit_eps, eps, out_scale, state, conv,
            segments.row0, segments.rows, segments.slot, segments.longest,
            row_seq, ctx, segments.longs, segments.chunks, segments.SHORT,
            out)
        return out
    return torch_ref.channel_delta(
        ab, ag, heads, kv_heads, dp, vp, dim, vdim, conv_w, a_log, dt_bias,
        o_norm, unit_eps, eps, out_scale, state, conv, segments, row_seq,
        ctx, out)


def lru_gate_order(w):
    """Gate weights [.., out, in] in the order in which the MFMA takes them
    (32 outputs by 32 inputs at a time), in the same shape; sizes % 32."""
    n = w.shape[-1]
    t = w.reshape(-1, n // 32, 16, 2, n // 32, 4, 8)
    return t.permute(0, 1, 4, 3, 5, 2, 6).reshape(w.shape)


def gated_lru(ab, conv_w, conv_b, gates, gates_b, decay, state, conv,
              segments, row_seq, ctx, chunk):
    """Linear recurrent unit of a ragged step on the projection ab [M,
    GELU branch | recurrent branch]: convolution, block-diagonal gates,
    recurrence in fp32, times the GELU branch. -> [M, width]; state and
    convolution slots are updated. Long segments run in chunks of `chunk`
    rows."""
    if ab.is_cuda:
        _require_hip("_hip_lru")
        longs, chunks = segments.chunk_lists(chunk)
        return _hip_ops.gated_lru(
            ab, conv_w, conv_b, gates, gates_b, decay, state, conv,
            segments.row0, segments.rows, segments.slot, segments.longest,
            row_seq, ctx, longs, chunks, chunk, segments.SHORT)
    return torch_ref.gated_lru(ab, conv_w, conv_b, gates, gates_b, decay,
                               state, conv, segments, row_seq, ctx)


# ---- retention / rotary latent attention decoder on several streams ---------

def stream_step(x, y=None, writes=None, mix=None, shared=None, embed=None,
                read=None, norm=None, store=True, dtype=None):
    """One boundary of fp32 residual streams x [M, S, W], in place. With a
    sublayer's output y [M, W] and writes = (out [S], then the matrix mix,
    from-major), x_t becomes sum_s mix[s, t] x_s + out[t] y. With mix
    [M, top] (+ 1 column with shared [M, W]), y [M * top, W] is summed with
    these weights first. With embed = (tokens, table) every old stream is
    the token's row and x is not read; without `store` x is not written.
    Returns rms(sum_s read[s] x_s) * w (read None: the plain sum) with norm
    = (w, n, eps), statistics over n columns, in `dtype` (default: y's)."""
    w, n, eps = norm
    if dtype is None:
        dtype = y.dtype
    if x.is_cuda:
        _require_hip("_hip_residual")
        tokens, table = embed if embed is not None else (None, None)
        h = torch.empty(x.shape[0], x.shape[2], dtype=dtype, device=x.device)
        _hip_ops.stream_step(x, y, writes, mix, shared, tokens, table, read,
                             w, n, eps, store, h)
        return h
    return torch_ref.stream_step(x, y, writes, mix, shared, embed, read,
                                 norm, store, dtype)


def retention(ab, heads, dp, vp, dim, vdim, decay, table, eps, state,
              segments, ctx):
    """Linear attention with a fixed decay per head (decay [2, heads]: the
    decays, their base-2 logarithms) of a ragged step, on the projection
    ab [M, queries | keys | values | gates]: rotation by table, recurrence
    in fp32, heads normed over vdim and gated by silu. -> [M, heads * vp];
    the sequences' slots of state [slots, heads, vp, dp] are updated."""
    if ab.is_cuda:
        _require_hip("_hip_retention")
        return _hip_ops.retention(
            ab, heads, dp, vp, dim, vdim, decay, table, eps, state,
            segments.row0, segments.rows, segments.slot, ctx,
            *segments.pieces(heads), segments.SHORT)
    return torch_ref.retention(ab, heads, dp, vp, dim, vdim, decay, table,
                               eps, state, segments, ctx)
