"""Paged decode attention at the edges of pages, 32-key tiles, waves and
shares of a sequence, for every number of query heads per key head; the launch
that rotates and stores a step's projections."""

from __future__ import annotations

import math

import pytest
import torch

from distllm_amd import ops
from distllm_amd.ops import torch_ref

pytestmark = pytest.mark.gpu


def _pages(B, HKV, D, lens, width, fp8, seed, device, stale=float("nan")):
    """Pages in mixed order; rows behind a sequence's end hold `stale`."""
    g = torch.Generator().manual_seed(seed)
    n = B * width + 1
    k = torch.randn(n, HKV, 16, D, generator=g)
    v = torch.randn(n, HKV, 16, D, generator=g)
    table = (torch.randperm(n - 1, generator=g) + 1).int().view(B, width)
    for b, L in enumerate(lens):
        if L % 16:
            for t in (k, v):
                t[table[b, L // 16], :, L % 16:] = stale
    if fp8:
        k, v = (t.to(torch.float8_e4m3fn) for t in (k, v))
    else:
        k, v = (t.to(torch.bfloat16) for t in (k, v))
    return k.to(device), v.to(device), table.to(device)


def _want(q, k, v, table, lens, scale):
    """In fp32 on the host, as bf16 products are not safe there."""
    out = torch.zeros(q.shape)
    k, v, table = (t.cpu() for t in (k.float(), v.float(), table))
    rep = q.shape[1] // k.shape[1]
    for b, L in enumerate(lens):
        if L == 0:
            continue
        pages = table[b, : -(-L // 16)].long()
        kk, vv = (t[pages].transpose(0, 1).reshape(k.shape[1], -1, k.shape[3])
                  [:, :L].repeat_interleave(rep, 0) for t in (k, v))
        s = (kk @ q[b].float().cpu()[..., None])[..., 0] * scale
        out[b] = (s.softmax(-1)[:, None] @ vv)[:, 0]
    return out


# bf16 results of fp32 sums
TOL = {"atol": 2e-3, "rtol": 8e-3}


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H,HKV", [(4, 4), (6, 2), (8, 1), (10, 2), (20, 1),
                                   (32, 8)])
def test_forms(device, H, HKV, D, fp8):
    lens = [1, 15, 16, 17, 31, 32, 33, 127, 128, 129, 300, 0]
    k, v, table = _pages(len(lens), HKV, D, lens, 20, fp8, H * D, device,
                         float("nan"))
    q = torch.randn(len(lens), H, D, device=device).to(torch.bfloat16)
    raw = [t.view(torch.uint8) if fp8 else t for t in (k, v)]
    ctx = torch.tensor(lens, dtype=torch.int32, device=device)
    out = ops.paged_attn(q, *raw, table, ctx)
    torch.testing.assert_close(out.float().cpu(),
                               _want(q, k, v, table, lens, D ** -0.5), **TOL)


@pytest.mark.parametrize("B,width,lens", [
    (1, 300, [4800]), (1, 300, [33]), (2, 64, [1024, 5]), (1, 1100, [17600]),
    (3, 40, [640, 639, 500])])
def test_shares(device, B, width, lens):
    k, v, table = _pages(B, 2, 128, lens, width, False, width, device)
    q = torch.randn(B, 8, 128, device=device).to(torch.bfloat16)
    ctx = torch.tensor(lens, dtype=torch.int32, device=device)
    for scale in (0.1, -0.3):
        out = ops.paged_attn(q, k, v, table, ctx, scale)
        torch.testing.assert_close(out.float().cpu(),
                                   _want(q, k, v, table, lens, scale), **TOL)


def test_probabilities_in_32_bits(device):
    """One large score and many small ones: what 16-bit probabilities would
    lose in their sum is more than a bf16 step of the result."""
    L, D = 4096, 64
    k, v, table = _pages(1, 1, D, [L], L // 16, False, 3, device)
    q = torch.randn(1, 1, D, device=device).to(torch.bfloat16)
    ctx = torch.tensor([L], dtype=torch.int32, device=device)
    out = ops.paged_attn(q, k, v.fill_(1.0), table, ctx)
    assert (out == 1).all()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("H,HKV,D", [(4, 2, 64), (32, 8, 128), (3, 3, 128)])
@pytest.mark.parametrize("B", [1, 5])
def test_rope_put(device, B, H, HKV, D, fp8):
    lens = [1, 16, 17, 40, 63][:B]
    k, v, table = _pages(B, HKV, D, lens, 4, fp8, B, device, 0.0)
    raw = [t.view(torch.uint8) if fp8 else t for t in (k, v)]
    old = [t.clone() for t in raw]
    cs, sn = ops.rope_tables(64, D, device=device)
    qkv = torch.randn(B, H + 2 * HKV, D, device=device).to(torch.bfloat16)
    ctx = torch.tensor(lens, dtype=torch.int32, device=device)
    q = ops.rope_put(qkv, cs, sn, ctx, *raw, table)
    rot = ops.rope_apply(qkv, cs, sn, ctx - 1, rope_heads=H + HKV)
    torch.testing.assert_close(q, rot[:, :H], atol=0, rtol=2 ** -7)
    ops.cache_put(rot[:, H: H + HKV].contiguous(),
                  rot[:, H + HKV:].contiguous(), *old, table, ctx - 1)
    for got, want in zip(raw, old):
        if fp8:  # a neighbouring number where the rotation rounds otherwise
            assert (got.int() - want.int()).abs().max() <= 1
        else:
            torch.testing.assert_close(got, want, atol=0, rtol=2 ** -7)
