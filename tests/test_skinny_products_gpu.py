"""Products of few rows in every form (direct, ring, tile, shared K) at the
edges of their ranges, with every activation."""

from __future__ import annotations

import pytest
import torch

from distllm_amd import ops
from distllm_amd.ops import torch_ref

pytestmark = pytest.mark.gpu

ROWS = [1, 2, 3, 15, 16, 17, 32, 33, 64, 65, 128, 129, 256]
# least sizes; K of one, of fewer chunks than waves or buffers, of odd
# chunk counts; columns that change the form at 17 to 32 rows
SIZES = [(64, 64), (64, 192), (192, 320), (768, 768), (128, 3072),
         (8192, 256), (8320, 448)]


def _inputs(M, N, K, device, seed):
    g = torch.Generator(device=device).manual_seed(seed)

    def some(*s):
        return torch.randn(*s, device=device, generator=g).to(torch.bfloat16)

    return some(M, K), some(N, K) * K ** -0.5, some(N)


def _close(out, ref):
    # both sides sum in fp32; what is left is the rounding of the result
    # (2^-9 of it) and of sums that cancel
    torch.testing.assert_close(out.float(), ref, atol=4e-3, rtol=8e-3)


@pytest.mark.parametrize("N,K", SIZES)
@pytest.mark.parametrize("M", ROWS)
def test_forms(device, M, N, K):
    x, w, b = _inputs(M, N, K, device, M * N + K)
    ref = x.float() @ w.float().T
    _close(ops._hip_ops.decode_gemm(x, w, None, 0), ref)
    _close(ops._hip_ops.decode_gemm(x, w, b, 0), ref + b.float())
    for share in (1, 2, 5):
        if K % (64 * share) == 0:
            _close(ops._hip_ops.decode_gemm(x, w, b, share), ref + b.float())


@pytest.mark.parametrize("M", [1, 2, 9, 24, 48, 100, 200])
@pytest.mark.parametrize("share", [0, 2])
def test_activations(device, M, share):
    N, K = 256, 512
    x, w, b = _inputs(M, N, K, device, M)
    z = x.float() @ w.float().T
    zb = z + b.float()
    gate, up = zb[:, : N // 2], zb[:, N // 2:]
    act = torch.tensor([0.3, -0.2], device=device)
    F = torch.nn.functional
    run = ops._hip_ops.decode_gemm
    _close(run(x, w, b, share, 1), F.silu(gate) * up)
    _close(run(x, w, b, share, 2, 1.1, 1.702, 1.0),
           torch_ref.clamped_glu(zb, 1.1, 1.702, 1.0).float())
    _close(run(x, w, b, share, 3, act_nums=act), torch_ref.xielu(zb, act))
    _close(run(x, w, b, share, 5), F.relu(zb) ** 2)
    _close(run(x, w, b, share, 6), F.gelu(zb, approximate="tanh"))
    _close(run(x, w, b, share, 7), F.gelu(zb))
    _close(run(x, w, b, share, 8), F.silu(zb))
    table = torch.randn(11, 300, device=device).to(torch.bfloat16)
    tokens = torch.arange(M, device=device) % 11
    rows = torch.zeros(M, N, device=device)
    rows[:, :200] = (F.gelu(z, approximate="tanh")[:, :200]
                     * table.float()[tokens, 30:230])
    _close(ops._hip_ops.decode_gemm_rows(x, w, share, tokens, table, 30, 200),
           rows)


@pytest.mark.parametrize("M", [17, 32, 33, 64])
@pytest.mark.parametrize("N, K, shares", [
    (12288, 512, 1), (16384 + 3072, 576, 1), (27648, 512, 1), (32768, 640, 1),
    (6144, 2048, 2), (5120, 2048, 2), (6144, 1024, 2),
    (12288, 1536, 1), (12288, 2560, 1), (19456, 768, 1), (19456, 1088, 1),
    (24576, 768, 1), (24576, 1600, 1), (28672, 2560, 1), (27648, 2624, 1),
    (32768, 3072, 1), (32768, 4096, 1), (5632, 1024, 2), (5120, 4096, 4),
    (5632, 4096, 4), (6144, 4096, 4), (2560, 8192, 8), (3072, 12288, 8)])
def test_columns_even_on_the_card(device, M, N, K, shares):
    """48 to 128 columns a workgroup, all and some with one block less, of one
    share and of several, with the least sums that take them, and short ones
    that do not."""
    run, F = ops._hip_ops.decode_gemm, torch.nn.functional
    assert ops._hip_ops.decode_gemm_shares(M, N, K) == shares
    x, w, b = _inputs(M, N, K, device, M + N)
    z = x.float() @ w.float().T
    zb = z + b.float()
    _close(run(x, w, None, 0), z)
    _close(run(x, w, b, 0), zb)
    torch.testing.assert_close(run(x, w, b, 0, 9), run(x, w, b, 0).float(),
                               atol=0, rtol=0)
    _close(run(x, w, b, 0, 1), F.silu(zb[:, : N // 2]) * zb[:, N // 2:])
    _close(run(x, w, b, 0, 2, 1.1, 1.702, 1.0),
           torch_ref.clamped_glu(zb, 1.1, 1.702, 1.0).float())
    if shares > 1:
        _close(ops._hip_ops.decode_gemm_parts(x, w).sum(0), z)


@pytest.mark.parametrize("N, K", [(64, 2048), (192, 2112), (1024, 4096),
                                  (1984, 2048), (2048, 2240)])
@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 25, 32, 33, 41, 49, 57, 64])
def test_eight_columns(device, M, N, K):
    """Up to 2048 columns with sums that begin in turn."""
    x, w, b = _inputs(M, N, K, device, M + N)
    z = x.float() @ w.float().T
    _close(ops._hip_ops.decode_gemm(x, w, None, 0), z)
    _close(ops._hip_ops.decode_gemm(x, w, b, 0), z + b.float())


@pytest.mark.parametrize("M", [1, 8, 24, 64])
@pytest.mark.parametrize("N, K", [(64, 2048), (1024, 4096), (2048, 2176),
                                  (2112, 2048)])
def test_sums_are_in_one_order(device, M, N, K):
    """Of 8 columns a workgroup (up to 2048) as of 16, which a 32-bit result and
    a row with its norm ahead have: of products that cancel each other what is
    left are the roundings on the way."""
    g = torch.Generator(device=device).manual_seed(N + K + M)

    def randn(*shape):
        return torch.randn(*shape, device=device, generator=g).bfloat16()

    def twice(t, sign=1):
        return torch.cat((t, sign * t.flip(-1)), -1).contiguous()

    w = randn(N, K // 2) * 2.0 ** torch.randint(0, 12, (N, K // 2),
                                                device=device, generator=g)
    w = twice(w.bfloat16(), -1)
    x = twice(randn(M, K // 2))
    want = ops.linear(x, w)
    assert want.any()
    assert torch.equal(ops.linear_f32(x, w), want.float())
    if M == 1:
        a, nw = twice(randn(1, K // 2)), twice(randn(K // 2))
        got, _ = ops.norm_linear(a, x, nw, 1e-5, w)
        h, _ = ops.norm_fwd_sum(a, x, nw, rms=True)
        assert torch.equal(got, ops.linear(h, w))


def test_refusals(device):
    x, w, _ = _inputs(4, 128, 128, device, 1)
    for args in ((x, w, None, 1, 1), (x, w, None, 3), (x, w, None, 0, 4),
                 (x, w[:96], None, 0), (x[:, :96].contiguous(),
                                        w[:, :96].contiguous(), None, 0)):
        with pytest.raises(RuntimeError):
            ops._hip_ops.decode_gemm(*args)


@pytest.mark.parametrize("act", [ops.ACT_NONE, ops.ACT_GELU_TANH,
                                 ops.ACT_GELU_ERF, ops.ACT_SILU])
@pytest.mark.parametrize("M", [1, 24, 128, 130])
def test_linear(device, M, act):
    x, w, b = _inputs(M, 192, 256, device, M)
    _close(ops.linear(x[None], w, b, act)[0],
           torch_ref.gemm(x.float(), w.float(), b.float(), act).float())


@pytest.mark.parametrize("act", [ops.ACT_GELU_ERF, ops.ACT_SILU])
def test_strided_weights(device, act):
    """Weights and biases that the form does not read as they lie."""
    x, w, b = _inputs(20, 192, 256, device, 5)
    want = torch_ref.gemm(x.float(), w.float(), b.float(), act).float()
    _close(ops.linear(x, w.t().contiguous().t(), b, act), want)
    _close(ops.linear(x, w, torch.stack([b, b], 1)[:, 0], act), want)
    wide = torch.zeros(20, 257, device=device, dtype=torch.bfloat16)
    wide[:, 1:] = x
    _close(ops.linear(wide[:, 1:], w, b, act), want)


@pytest.mark.parametrize("mode", ["gemm8", "gemm16", "blaslt"])
@pytest.mark.parametrize("act", [ops.ACT_NONE, ops.ACT_GELU_ERF])
def test_forced_form(device, mode, act, monkeypatch):
    """A form that the caller asks for is not overruled for few rows of a
    product with an activation; without one the choice stays measured."""
    x, w, b = _inputs(20, 192, 256, device, 5)
    calls, real = [], ops._hip_ops

    class Spy:
        def __getattr__(self, name):
            if name == "decode_gemm":
                calls.append(name)
            return getattr(real, name)

    monkeypatch.setenv("DISTLLM_GEMM", mode)
    monkeypatch.setattr(ops, "_hip_ops", Spy())
    monkeypatch.setattr(ops, "_GEMM_CHOICE", {})
    out = ops.linear(x, w, b, act)
    _close(out, torch_ref.gemm(x.float(), w.float(), b.float(), act).float())
    assert not calls or (act == ops.ACT_NONE and mode != "blaslt")
    measured = bool(ops._GEMM_CHOICE)
    assert measured == (act == ops.ACT_NONE and mode != "blaslt")


@pytest.mark.parametrize("act", [ops.ACT_NONE, ops.ACT_GELU_ERF])
@pytest.mark.parametrize("M", [1, 20, 100])
def test_bias_sizes(device, M, act):
    """A bias that is not one number per column is refused, or spread, by the
    library's product, whose rules hold for every number of rows."""
    x, w, b = _inputs(M, 192, 256, device, 5)
    for wrong in (b[:100].contiguous(), b[:0].contiguous(), b.cpu()):
        with pytest.raises(RuntimeError):
            ops.linear(x, w, wrong, act)
        with pytest.raises(RuntimeError):
            ops._hip_ops.decode_gemm(x, w, wrong, 0)
    want = torch_ref.gemm(x.float(), w.float(), b[:1].float().expand(192),
                          act).float()
    _close(ops.linear(x, w, b[:1].contiguous(), act), want)


@pytest.mark.parametrize("M", [1, 8, 9, 16, 17])
@pytest.mark.parametrize("N,K", [(16320, 128), (16384, 128), (16384, 1024),
                                 (16384, 1088), (16448, 1536), (16384, 1600)])
def test_short_sums(device, M, N, K):
    """Both sides of where up to 16 rows leave the ring."""
    x, w, b = _inputs(M, N, K, device, M * N + K)
    ref = x.float() @ w.float().T + b.float()
    _close(ops.linear(x, w, b), ref)
    _close(ops.linear(x, w, b, ops.ACT_GELU_ERF),
           torch.nn.functional.gelu(ref))


def test_vocabulary(device, monkeypatch):
    """The choice for wide products without an activation is measured."""
    monkeypatch.setattr(ops, "_GEMM_CHOICE", {})
    for M, N, K, measured in ((16, 32832, 1536, 0), (17, 32768, 1536, 0),
                              (17, 32832, 1472, 0), (17, 32832, 1536, 1),
                              (64, 32832, 1536, 1)):
        x, w, b = _inputs(M, N, K, device, M)
        _close(ops.linear(x, w, b), x.float() @ w.float().T + b.float())
        assert len(ops._GEMM_CHOICE) == measured
        ops.linear(x, w, b, ops.ACT_SILU)
        assert len(ops._GEMM_CHOICE) == measured


@pytest.mark.parametrize("act", [ops.ACT_NONE, ops.ACT_GELU_ERF])
@pytest.mark.parametrize("M, N", [(0, 128), (5, 0), (0, 0)])
def test_nothing_to_do(device, M, N, act):
    x = torch.zeros(M, 128, device=device, dtype=torch.bfloat16)
    w = torch.zeros(N, 128, device=device, dtype=torch.bfloat16)
    assert ops._hip_ops.decode_gemm(x, w, None, 0).shape == (M, N)
    if N:
        assert ops.linear(x, w, None, act).shape == (M, N)
        assert ops.gateup_swiglu(x, w).shape == (M, N // 2)
    torch.cuda.synchronize()


def test_vocabulary_in_a_capture(device, monkeypatch):
    """A wide product that was never measured can be captured."""
    monkeypatch.setattr(ops, "_GEMM_CHOICE", {})
    monkeypatch.setattr(ops, "_WIDE_RUN", set())
    ops.linear(*_inputs(20, 64, 128, device, 0))
    x, w, b = _inputs(20, 32832, 1536, device, 5)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.linear(x, w, b)
    assert not ops._GEMM_CHOICE
    for seed in range(3):
        x.copy_(_inputs(20, 64, 1536, device, seed)[0])
        graph.replay()
        torch.cuda.synchronize()
        _close(out, x.float() @ w.float().T + b.float())
