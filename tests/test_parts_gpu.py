"""Products whose shares of K the next kernel sums: against the summed product
and the same kernels on it."""
import pytest
import torch

from distllm_amd import ops

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _rand(*shape, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*shape, device="cuda", generator=g).to(BF16)


@pytest.mark.parametrize("M", [1, 16, 17, 33, 64, 65])
@pytest.mark.parametrize("N, K", [(4096, 14336), (1024, 4096), (8192, 1536),
                                  (4160, 768)])
def test_norm(device, M, N, K):
    x, w, res = _rand(M, K), _rand(N, K, seed=1), _rand(M, 1, N, seed=2)
    nw = _rand(N, seed=3)
    got, total = ops.norm_parts_sum(ops.linear_parts(x, w), res, nw)
    want, sums = ops.norm_fwd_sum(ops.linear(x, w).view_as(res), res, nw,
                                  rms=True)
    assert torch.equal(total, sums) and got.shape == res.shape
    # the squares are summed in another order: the last of bf16's 7 bits
    torch.testing.assert_close(got, want, rtol=2 ** -7, atol=1e-6)


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("cache", ["bf16", "fp8"])
@pytest.mark.parametrize("B, H, HKV, D, K", [
    (1, 32, 8, 128, 4096), (17, 32, 8, 128, 4096), (64, 32, 8, 128, 4096),
    (40, 3, 1, 64, 8192), (64, 5, 2, 128, 3072)])
def test_rope_put(device, B, H, HKV, D, K, cache, bias):
    heads = H + 2 * HKV
    x, w = _rand(B, K), _rand(heads * D, K, seed=1)
    b = _rand(heads * D, seed=2) * 30 if bias else None
    cs, sn = (torch.randn(300, D // 2, device="cuda") for _ in range(2))
    ctx = torch.randint(1, 300, (B,), device="cuda", dtype=torch.int32)
    bt = torch.arange(B * 19, dtype=torch.int32, device="cuda").view(B, 19)
    out = []
    for f in (ops.linear, ops.linear_parts):
        kc, vc = (torch.zeros(B * 19, HKV, 16, D, device="cuda", dtype=BF16
                              if cache == "bf16" else torch.uint8)
                  for _ in range(2))
        qkv = f(x, w, b)
        q = ops.rope_put(qkv.view(*qkv.shape[:-1], heads, D), cs, sn, ctx, kc,
                         vc, bt, b)
        out.append((q, kc, vc))
    assert all(torch.equal(a, c) for a, c in zip(*out))
    assert out[0][1].any() and out[0][2].any()


def test_shares_taken(device):
    """Slabs where K is shared, the product elsewhere."""
    w = _rand(4096, 4096)
    assert ops.linear_parts(_rand(64, 4096), w).dim() == 3
    assert ops.linear_parts(_rand(16, 4096), w).dim() == 2
    assert ops.linear_parts(_rand(65, 4096), w).dim() == 2


@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("N, K", [(128, 1280), (1152, 1344), (256, 2048),
                                  (384, 2560), (6144, 4096), (128, 4160),
                                  (256, 8192), (128, 1216)])
def test_norm_linear(device, rows, gated, N, K):
    """Norm and product in one launch, bit for bit as in two, at the ends of
    its range and outside."""
    a, b = _rand(rows, K), _rand(rows, 1, K, seed=1)
    w, nw = _rand(N, K, seed=2), _rand(K, seed=3)
    bias = None if gated else _rand(N, seed=4) * 9
    got, x = ops.norm_linear(a, b, nw, 1e-5, w, bias, gated)
    h, want_x = ops.norm_fwd_sum(a.view_as(b), b, nw, rms=True)
    want = (ops.gateup_swiglu(h[:, 0], w) if gated
            else ops.linear(h[:, 0], w, bias))
    assert torch.equal(x, want_x) and torch.equal(got, want)


@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("N, K", [(32, 2560), (1040, 2688), (6144, 4096),
                                  (24, 4224), (256, 8192), (64, 2432),
                                  (64, 2576)])
def test_norm_linear_fp8(device, rows, gated, N, K):
    if gated and K % 128:
        N = 64  # the gated unit of other K is a kernel of its own
    a, b = _rand(rows, K), _rand(rows, 1, K, seed=1)
    nw, scale = _rand(K, seed=3), torch.rand(N, device="cuda") + 0.1
    w = _rand(N, K, seed=2).to(torch.float8_e4m3fn).view(torch.uint8)
    bias = None if gated else _rand(N, seed=4) * 9
    got, x = ops.norm_linear_fp8(a, b, nw, 1e-5, w, scale, bias, gated)
    h, want_x = ops.norm_fwd_sum(a.view_as(b), b, nw, rms=True)
    want = (ops.gateup_swiglu_fp8(h[:, 0], w, scale) if gated
            else ops.gemv_fp8(h[:, 0], w, scale, bias))
    assert torch.equal(x, want_x) and torch.equal(got, want)


@pytest.mark.parametrize("rows", [1, 2, 8])
@pytest.mark.parametrize("K", [2560, 2432, 2576])
def test_gated_bias_fp8(device, rows, K):
    """The bias of a quantized gated unit, in one launch, in two, and at a K
    that the ring form does not take."""
    N = 64
    a, b = _rand(rows, K), _rand(rows, 1, K, seed=1)
    nw, scale = _rand(K, seed=3), torch.rand(N, device="cuda") * 0.01 + 0.01
    w = _rand(N, K, seed=2).to(torch.float8_e4m3fn)
    bias = _rand(N, seed=4) * 9
    got, _ = ops.norm_linear_fp8(a, b, nw, 1e-5, w.view(torch.uint8), scale,
                                 bias, True)
    h, _ = ops.norm_fwd_sum(a.view_as(b), b, nw, rms=True)
    z = (h[:, 0].double() @ w.double().T * scale.double() + bias.double())
    want = torch.nn.functional.silu(z[:, : N // 2]) * z[:, N // 2:]
    # the output's bf16, and at other K that of gate and up before the product
    torch.testing.assert_close(got.double(), want, rtol=2 ** -6, atol=2e-2)


@pytest.mark.parametrize("M", [17, 32])
@pytest.mark.parametrize("N, K, shares", [(4096, 4096, 4), (2048, 4096, 8),
                                          (2048, 4032, 1), (4096, 2048, 4)])
def test_shares_in_place_of_the_ring(device, M, N, K, shares):
    """Products that a launch of their own would not share K for."""
    x, w = _rand(M, K), _rand(N, K, seed=1)
    assert ops._hip_ops.decode_gemm_shares(M, N, K) == 1
    got = ops.linear_parts(x, w)
    assert got.shape == ((shares, M, N) if shares > 1 else (M, N))
    want = x.double() @ w.double().t()
    total = (got.sum(0) if shares > 1 else got).double()
    bound = (x.double().abs() @ w.double().abs().t()) * K * 2 ** -24
    if shares == 1:
        bound += want.abs() * 2 ** -8
    assert ((total - want).abs() <= bound).all()


@pytest.mark.parametrize("M", [1, 16, 17, 32, 33, 64, 65])
@pytest.mark.parametrize("N, K", [(4096, 4096), (2048, 4096), (6144, 2048),
                                  (768, 768), (1024, 8192)])
def test_shares_joined(device, M, N, K):
    """The slabs' sum, one after the other, rounded once."""
    x, w = _rand(M, K), _rand(N, K, seed=1)
    parts = ops.linear_parts(x, w)
    total = parts if parts.dim() == 2 else torch.zeros_like(parts[0])
    for p in parts if parts.dim() == 3 else ():
        total += p
    assert torch.equal(ops.linear_joined(x, w), total.to(BF16))


@pytest.mark.parametrize("S", [2, 3, 8])
@pytest.mark.parametrize("QP, qn, R, rn", [(128, 100, 192, 130),
                                           (1536, 1536, 512, 512),
                                           (4096, 4000, 2112, 2100)])
def test_latent_prep(device, S, QP, qn, R, rn):
    """Both norms of the sum of slabs against those of the sum in bf16; a row
    without a place in the cache writes nothing."""
    M = 5
    ab = torch.randn(S, M, QP + R, device="cuda")
    ab[:, :, qn:QP] = 0
    ab[:, :, QP + rn:] = 0
    wq, wc = torch.randn(QP, device="cuda"), torch.randn(R, device="cuda")
    bt = torch.tensor([[3, 1, 0], [5, 2, 4]], dtype=torch.int32, device="cuda")
    seq = torch.tensor([0, 0, 1, 0, 1], dtype=torch.int32, device="cuda")
    ctx = torch.tensor([40, 17, 7, 0, 1], dtype=torch.int32, device="cuda")
    total = ab[0].clone()
    for s in range(1, S):
        total += ab[s]
    out = []
    for x in (ab, total.to(BF16)):
        cache = torch.zeros(6, 16, R, dtype=BF16, device="cuda")
        cq = ops.latent_prep(x, QP, qn, rn, wq, wc, 1e-3, cache, bt, seq, ctx)
        out.append((cq, cache))
    for a, b in zip(*out):
        # the squares are summed in another order: the last of bf16's 7 bits
        torch.testing.assert_close(a, b, rtol=2 ** -7, atol=1e-6)
        assert torch.equal(a == 0, b == 0)
    alone = ops.latent_prep(ab[:, :, :QP].contiguous(), QP, qn, rn, wq, None,
                            1e-3, None, bt, seq, ctx)
    assert torch.equal(alone, out[0][0])
    with pytest.raises(RuntimeError):
        ops.latent_prep(ab, QP, qn, rn, wq, wc, 1e-3, cache.float(), bt, seq,
                        ctx)
