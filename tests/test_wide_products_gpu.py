"""Products of many rows (csrc/wide_gemm.hip): tiles, remainders, activations
and units against fp32 references, and which calls linear sends there."""

import pytest
import torch
import torch.nn.functional as F

import distllm_amd.ops as ops

pytestmark = pytest.mark.gpu


def _operands(M, N, K, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    b = torch.randn(N, device="cuda", generator=g).bfloat16()
    return x, w, b


def _reference(x, w, b, act):
    y = x.double() @ w.double().T
    if b is not None:
        y = y + b.double()
    if act == ops.ACT_GELU_TANH:
        return F.gelu(y, approximate="tanh")
    if act == ops.ACT_GELU_ERF:
        return F.gelu(y)
    if act == ops.ACT_SILU:
        return F.silu(y)
    if act >= 4:
        g, u = y.chunk(2, 1)
        if act == 4:
            return F.silu(g) * u
        g, u = g.clamp(max=1.5), u.clamp(-1.5, 1.5)
        return g * torch.sigmoid(1.702 * g) * (u + 1)
    return y


def _check(got, want):
    # the result's rounding to 8 bits, and sums of at most 1024 terms of size
    # 1 in 32 bits ahead of an activation whose slope is below 2 x its factor
    bound = want.abs() * 2.0 ** -8 + 2e-5 * (1 + want.abs().amax())
    assert ((got.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("tile", [4, 5, 6, 7, 8])
@pytest.mark.parametrize("M,N,K", [
    (1, 256, 128),      # one row of one tile, two stages
    (257, 512, 192),    # a row behind a tile's edge, an odd count of stages
    (2049, 768, 128),   # more row tiles than go together, some in the last
    (9001, 2304, 256),  # workgroups with more tiles than one
    (300, 256, 1024),   # more stages than slots, a few times
])
def test_tiles(tile, M, N, K):
    x, w, b = _operands(M, N, K)
    _check(ops._hip_ops.wide_gemm(x, w, b, 0, tile), _reference(x, w, b, 0))


@pytest.mark.parametrize("tile", [4, 6, 8])
@pytest.mark.parametrize("M,N,K,act", [
    (1100, 512, 4096, 0), (300, 512, 14336, 0), (2100, 4096, 4096, 0),
    (1100, 1024, 4096, 4), (300, 512, 14336, 2)])
def test_long_sums(tile, M, N, K, act):
    """K of a decoder's products, with one round of tiles and several. Errors
    of the terms' sums are as steps at random, sqrt(K) 2^-24 of 4 or so: 3e-5."""
    x, w, b = _operands(M, N, K)
    got = ops._hip_ops.wide_gemm(x, w, b, act, tile)
    want = _reference(x, w, b, act)
    bound = want.abs() * 2.0 ** -8 + 6e-5 * (1 + want.abs().amax())
    assert ((got.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("act", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("M,tile", [(70, 8), (4099, 6)])
def test_ends(act, bias, M, tile):
    x, w, b = _operands(M, 1024, 320)
    b = b if bias else None
    got = ops._hip_ops.wide_gemm(x, w, b, act, tile, 1.5, 1.702, 1.0)
    _check(got, _reference(x, w, b, act))


def test_large_result():
    """Above 256 MiB the result is written past the caches."""
    x, w, b = _operands(46000, 3072, 128)
    got = ops._hip_ops.wide_gemm(x, w, b, 0, 8)
    at = torch.arange(0, 46000, 97, device="cuda")
    _check(got[at], _reference(x[at], w, b, 0))
    _check(got[-300:], _reference(x[-300:], w, b, 0))


def test_gelu_of_large_and_not_finite():
    x, w, b = _operands(300, 256, 128)
    x[:, 0], w[:, 1:] = 1.0, 0.0
    special = torch.tensor([float("inf"), float("nan"), 3e38, 80.0, 9.0, 5.5,
                            4.0, 1e-3, 1e-30, 0.0, -1e-3, -4.0, -5.5, -9.0,
                            -80.0, -3e38], device="cuda").bfloat16()
    w[:, 0] = 0
    b[:] = special.repeat(16)
    got = ops._hip_ops.wide_gemm(x, w, b, 2, 8).double()
    want = F.gelu(b.double()).expand(300, -1)
    assert torch.equal(got.isnan(), want.isnan())
    ok = ~want.isnan()
    same = got[ok] == want[ok]  # infinities among them
    close = (got[ok] - want[ok]).abs() <= want[ok].abs() * 2.0 ** -8 + 1e-6
    assert (same | close).all()


def test_gelu_of_small_results():
    """To the rounding of the result, half a unit of its eighth bit, also where
    little is left of x: 4e-4 of results above 1e-4 and 3e-7 are the function's
    own."""
    x, w, b = _operands(300, 2048, 128)
    x[:], w[:] = 1.0, 0.0
    b[:] = torch.linspace(-4.2, 9, 2048, device="cuda")
    got = ops._hip_ops.wide_gemm(x, w, b, ops.ACT_GELU_ERF, 8).double()
    want = F.gelu(b.double())
    half = torch.ldexp(torch.ones_like(want), want.frexp().exponent - 9)
    assert ((got - want).abs() <= half + want.abs() * 4e-4 + 3e-7).all()


@pytest.mark.parametrize("act", [ops.ACT_GELU_TANH, ops.ACT_GELU_ERF,
                                 ops.ACT_SILU])
def test_activations_of_infinities(act):
    """As torch has them, NaN for minus infinity among them."""
    x, w, b = _operands(300, 256, 128)
    x[:], w[:] = 1.0, 0.0
    b[:] = torch.tensor([float("inf"), float("-inf"), float("nan"), 0.0],
                        device="cuda").repeat(64)
    got = ops._hip_ops.wide_gemm(x, w, b, act, 8).double()
    want = _reference(x, w, b, act)
    assert want[0, 1].isnan()
    torch.testing.assert_close(got, want, rtol=0, atol=0, equal_nan=True)


def test_linear_takes_it_and_gives_the_library_s_result(monkeypatch):
    """Over the forms that linear accepts: shapes with leading dimensions,
    strided inputs and biases, storage that starts between 16-byte pieces."""
    calls = []
    own = ops._hip_ops.wide_gemm
    monkeypatch.setattr(ops._hip_ops, "wide_gemm",
                        lambda *a: calls.append(a) or own(*a), raising=False)
    x, w, b = _operands(6000, 2304, 256)

    def same(x, w, b, wide):
        calls.clear()
        got = ops.linear(x, w, b)
        assert got.shape == (*x.shape[:-1], w.shape[0])
        assert bool(calls) == wide
        _check(got.reshape(-1, w.shape[0]),
               _reference(x.reshape(-1, x.shape[-1]), w, b, 0))

    with torch.no_grad():
        same(x, w, b, True)
        same(x.view(6, 1000, 256), w, None, True)
        same(torch.nn.Parameter(x), torch.nn.Parameter(w), b, True)
        wide = torch.randn(6000, 512, device="cuda").bfloat16()
        same(wide[:, :256], w, b, False if not wide[:, :256].is_contiguous()
             else True)
        same(wide.view(3000, 4, 256).transpose(0, 1), w, b, True)  # a copy
        same(x, w, torch.stack([b, b], 1)[:, 0], False)
        flat = torch.empty(6000 * 256 + 1, device="cuda").bfloat16()
        flat[1:] = x.reshape(-1)
        same(flat[1:].view(6000, 256), w, b, True)
        same(x[:300], w, b, False)
        monkeypatch.setenv("DISTLLM_GEMM", "blaslt")
        same(x, w, b, False)
        monkeypatch.delenv("DISTLLM_GEMM")
    # gradients are the library's
    w = torch.nn.Parameter(w)
    calls.clear()
    y = ops.linear(x[:5999], w, b)
    assert y.requires_grad and not calls
    y.float().sum().backward()
    assert w.grad is not None


def test_units_take_it():
    x, w, _ = _operands(3000, 6144, 256)
    with torch.no_grad():
        assert ops._wide_tile(x, w, None, 4)
        _check(ops.gateup_swiglu(x, w), _reference(x, w, None, 4))
        _check(ops.gateup_clamped_glu(x, w, 1.5, 1.702, 1.0),
               _reference(x, w, None, 5))


@pytest.mark.parametrize("M,N,K,shares", [
    (65, 64, 128, 1),      # a row behind a block's edge, two chunks
    (128, 192, 448, 1),    # fewer chunks and as many as a ring's
    (300, 768, 768, 1),
    (1000, 1280, 1280, 1),
    (129, 128, 512, 2),    # shares of K, joined by a second launch
    (200, 768, 3072, 4),
])
@pytest.mark.parametrize("act", [ops.ACT_NONE, ops.ACT_GELU_TANH,
                                 ops.ACT_GELU_ERF, ops.ACT_SILU])
@pytest.mark.parametrize("bias", [False, True])
def test_blocks_of_64_rows(M, N, K, shares, act, bias):
    x, w, b = _operands(M, N, K)
    b = b if bias else None
    _check(ops._hip_ops.mid_gemm(x, w, b, shares, ops._DECODE_ACT[act]),
           _reference(x, w, b, act))


def test_linear_of_some_hundred_rows(monkeypatch):
    """By blocks of 64 where they fit, with the general path's results."""
    calls = []
    own = ops._hip_ops.mid_gemm
    monkeypatch.setattr(ops._hip_ops, "mid_gemm",
                        lambda *a: calls.append(a) or own(*a), raising=False)
    with torch.no_grad():
        for M, N, K, act, mid in [(65, 768, 768, 0, True),
                                  (300, 2304, 768, 2, True),
                                  (200, 768, 3072, 0, True),
                                  (64, 768, 768, 0, False),
                                  (1000, 3840, 1280, 0, False),
                                  (300, 4096, 4096, 0, False),
                                  (300, 2304, 800, 0, False)]:
            x, w, b = _operands(M, N, K)
            calls.clear()
            _check(ops.linear(x, w, b, act), _reference(x, w, b, act))
            assert bool(calls) == mid
        x, w, b = _operands(4 * 50, 768, 768)
        strided = torch.cat([x, x], 1)[:, :768].view(4, 50, 768)
        calls.clear()
        _check(ops.linear(strided, w, b).view(200, 768),
               _reference(x, w, b, 0))
        assert bool(calls) == strided.reshape(200, 768).is_contiguous()
    w.requires_grad_()
    calls.clear()
    assert ops.linear(x, w, b).requires_grad or not calls


@pytest.mark.parametrize("mode", ["decode", "blaslt", "gemm8", "gemm16"])
@pytest.mark.parametrize("M", [65, 128, 200, 256])
@pytest.mark.parametrize("act", [ops.ACT_NONE, ops.ACT_GELU_ERF])
def test_forms_that_are_asked_for(monkeypatch, mode, M, act):
    """DISTLLM_GEMM holds where blocks of 64 rows and tiles are the rule."""
    calls = []
    for name in ("mid_gemm", "wide_gemm", "decode_gemm"):
        own = getattr(ops._hip_ops, name)
        monkeypatch.setattr(
            ops._hip_ops, name, lambda *a, own=own, name=name:
            calls.append(name) or own(*a), raising=False)
    monkeypatch.setattr(ops, "_GEMM_CHOICE", {
        ("dec", n, 768, 768, True): "blaslt" for n in (128, 256)})
    x, w, b = _operands(M, 768, 768)
    with torch.no_grad():
        ops.linear(x, w, b, act)
        assert calls == ["mid_gemm"]
        calls.clear()
        monkeypatch.setenv("DISTLLM_GEMM", mode)
        got = ops.linear(x, w, b, act)
    if act == ops.ACT_NONE:  # else the library's sums are rounded ahead of it
        _check(got, _reference(x, w, b, act))
    # (an activation has no form in a launch of decode_gemm here)
    assert calls == (["decode_gemm"] if (mode, act) == ("decode", 0) else [])


@pytest.mark.parametrize("M,N,K", [
    (66, 4096, 4096), (128, 4096, 4096), (100, 2048, 8192), (256, 1280, 5120)])
def test_shares_of_k_in_a_graph(M, N, K):
    """As a captured step of so many sequences has them, 32 chunks of 64 of K
    and more a share."""
    x, w, b = _operands(M, N, K)
    with torch.no_grad():
        shares = ops._mid_shares(x, w, b)
        assert shares > 1 and K // shares >= 2048
        forms = [lambda: ops.linear(x, w, b),
                 lambda: ops._hip_ops.mid_gemm(x, w, b, shares, 0)]
        for run in forms:
            want = run()
            # of K terms in 32 bits, whose errors add up as steps at random
            _check(want, _reference(x, w, b, 0))
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                got = run()
            for _ in range(3):
                got.zero_()
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(got, want)


def test_linear_under_autocast():
    """To half precision by torch, as ever; to bf16 it is the same product."""
    x, w, b = _operands(300, 768, 768)
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16):
        got = ops.linear(x, w, b)
    assert got.dtype == torch.float16
    with torch.no_grad():
        want = ops.linear(x, w, b)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert torch.equal(ops.linear(x, w, b), want)


@pytest.mark.parametrize("B", [66, 128])
def test_captured_step_of_some_hundred_sequences(B, monkeypatch):
    """A decoder's step, whose products of short K go by blocks of 64 rows and
    whose last one, of a long K, by the choice that the first run measured."""
    from distllm_amd.models import ModelDims, build_model

    calls = []
    own = ops._hip_ops.mid_gemm
    monkeypatch.setattr(ops._hip_ops, "mid_gemm",
                        lambda *a: calls.append(a[0].shape[1]) or own(*a),
                        raising=False)
    monkeypatch.setattr(ops, "_GEMM_CHOICE", {})
    torch.manual_seed(B)
    m = build_model(ModelDims(
        arch="llama", vocab_size=512, hidden_size=512, num_layers=2,
        num_heads=8, num_kv_heads=2, intermediate_size=4096,
        max_position_embeddings=256), device="cuda")
    cache = m.make_cache(4 * B + 1, 16, "bf16")
    table = torch.randperm(4 * B, device="cuda").int().view(B, 4) + 1
    ctx = torch.randint(1, 65, (B,), device="cuda").int()
    tokens = torch.randint(0, 512, (B,), device="cuda")
    want = m.decode_step(tokens, cache, table, ctx)
    assert 512 in calls and 4096 in calls
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = m.decode_step(tokens, cache, table, ctx)
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        m.decode_step(tokens, cache, table, ctx)


def test_in_a_graph():
    x, w, b = _operands(3000, 2304, 768)
    with torch.no_grad():
        want = ops.linear(x, w, b, act=ops.ACT_GELU_ERF)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = ops.linear(x, w, b, act=ops.ACT_GELU_ERF)
        for _ in range(3):
            got.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(got, want)
