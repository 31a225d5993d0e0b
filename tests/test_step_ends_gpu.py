"""What a decode step begins and ends with: rows of tokens, their norm and the shares
of its attention in one launch, and products that are stored as 32 bits."""

import pytest
import torch

from distllm_amd import ops

pytestmark = pytest.mark.gpu


def _randn(*shape, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*shape, device="cuda", generator=g,
                       dtype=torch.bfloat16)


@pytest.mark.parametrize("n", [8, 1280, 2056, 8192])
@pytest.mark.parametrize("rows", [1, 5, 64, 1025])
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
def test_step_begin(rows, n, dtype):
    layers, heads, kv, D, blocks, V = 3, 8, 2, 64, 9, 97
    emb, w = _randn(V, n), _randn(n, seed=1)
    g = torch.Generator().manual_seed(rows)
    tokens = torch.randint(-V, V, (rows,), generator=g, dtype=dtype).cuda()
    tokens[0], tokens[-1] = -V, V - 1
    ctx = torch.randint(1, blocks * 16 + 1, (rows,), generator=g).int().cuda()
    table = torch.randint(0, 50, (rows, blocks), generator=g).int().cuda()
    cache = torch.zeros(50, kv, 16, D, device="cuda", dtype=torch.bfloat16)
    x, h, plan = ops.step_begin(tokens, emb, w, 1e-5, layers, ctx, heads,
                                cache, table)
    want = ops.step_plan(layers, ctx, heads, cache, table)
    assert len(plan) == len(want) == layers
    for (a, za), (b, zb) in zip(plan, want):
        # the eighth number is nobody's, nor the second four of what is no share
        used = b[:, 0] >= 0
        assert torch.equal(a[:, :4], b[:, :4])
        assert torch.equal(a[used, 4:6], b[used, 4:6])
        assert torch.equal(a[:rows, 6], b[:rows, 6])
        assert torch.equal(za, zb)
    assert x.shape == h.shape == (rows, 1, n)
    assert torch.equal(x, emb[tokens.long()].unsqueeze(1))
    f = x.double()
    ref = f * torch.rsqrt(f.square().mean(-1, keepdim=True) + 1e-5) * w.double()
    # 8 bits are kept: up to 2^-8 of a number, and what fp32 adds to it
    assert ((h.double() - ref).abs() <= ref.abs() * (2 ** -8 + 2 ** -18)).all()


def test_step_begin_other_tables():
    """What the launch does not take goes by launches of their own."""
    cache = torch.zeros(4, 2, 16, 64, device="cuda", dtype=torch.bfloat16)
    ctx = torch.ones(2, device="cuda", dtype=torch.int32)
    table = torch.zeros(2, 1, device="cuda", dtype=torch.int32)
    tokens = torch.tensor([3, -1], device="cuda")
    wide = _randn(7, 128)
    for emb in (wide[:, :64], _randn(7 * 64 + 1)[1:].view(7, 64)):
        w = _randn(64, seed=1)
        x, h, plan = ops.step_begin(tokens, emb, w, 1e-5, 1, ctx, 4, cache,
                                    table)
        assert torch.equal(x[:, 0], emb[tokens]) and len(plan) == 1
        assert torch.equal(h, ops.rms_norm(x, w, eps=1e-5))


@pytest.mark.parametrize("M", [1, 16, 17, 48, 64, 65])
@pytest.mark.parametrize("N,K", [(64, 128), (4096, 1536), (16384, 1024),
                                 (32768, 4096), (1000, 256)])
def test_linear_f32(M, N, K):
    x, w = _randn(M, 1, K), _randn(N, K, seed=1)
    out = ops.linear_f32(x, w)
    assert out.dtype == torch.float32 and out.shape == (M, 1, N)
    assert torch.equal(out, ops.linear(x, w).float())


@pytest.mark.parametrize("rows", [1, 3])
@pytest.mark.parametrize("N,K", [(64, 1280), (8192, 4096), (512, 8192)])
def test_norm_linear_f32(rows, N, K):
    a, b = _randn(rows, K), _randn(rows, 1, K, seed=1)
    w_norm, w = _randn(K, seed=2), _randn(N, K, seed=3)
    out, x = ops.norm_linear(a, b, w_norm, 1e-5, w, f32=True)
    want, sums = ops.norm_linear(a, b, w_norm, 1e-5, w)
    assert out.dtype == torch.float32 and torch.equal(x, sums)
    assert torch.equal(out, want.float())


@pytest.mark.parametrize("rows", [1, 3])
def test_a_replaced_linear_sees_the_logits(rows, monkeypatch):
    """Of both ways to make them, one row's with the norm in its launch."""
    a, b = _randn(rows, 1280), _randn(rows, 1, 1280, seed=1)
    w_norm, w = _randn(1280, seed=2), _randn(512, 1280, seed=3)
    first = ops.norm_linear(a, b, w_norm, 1e-5, w, f32=True)
    last = ops.linear_f32(a, w)
    seen, own = [], ops.linear
    monkeypatch.setattr(ops, "linear", lambda x, w, *r, **k: seen.append(
        w) or own(x, w, *r, **k))
    for g, v in zip(first, ops.norm_linear(a, b, w_norm, 1e-5, w, f32=True)):
        assert torch.equal(g, v)
    assert torch.equal(last, ops.linear_f32(a, w))
    assert len(seen) == 2 and all(s is w for s in seen)
