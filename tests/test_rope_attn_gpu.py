"""Attention that rotates its queries as it reads them, against the rotation and the
attention as launches of their own."""

import pytest
import torch

from distllm_amd import ops

pytestmark = pytest.mark.gpu

TOP = 400  # positions of the tables


def _qkv(*shape):
    g = torch.Generator(device="cuda").manual_seed(sum(shape))
    return torch.randn(*shape, device="cuda", generator=g,
                       dtype=torch.bfloat16)


def _tables(D):
    return ops.rope_tables(TOP, D, 10000.0, device="cuda")


def _positions(n):
    g = torch.Generator(device="cuda").manual_seed(n)
    return torch.randint(0, TOP, (n,), device="cuda", generator=g,
                         dtype=torch.int32)


def _same(a, b):
    # the rotated queries are the same numbers, but for a sum of two products
    # that may be rounded once or twice: a unit of their 8 bits in few of them
    assert (a.float() - b.float()).abs().max() < 2 ** -5
    assert (a != b).float().mean() < 0.02


@pytest.mark.parametrize("S", [1, 31, 128, 129, 300])
@pytest.mark.parametrize("H,HKV,D", [(2, 2, 64), (4, 1, 64), (4, 2, 128)])
@pytest.mark.parametrize("causal,masked", [(False, True), (True, True),
                                           (True, False)])
@pytest.mark.parametrize("scale", [None, -0.05])
def test_padded(S, H, HKV, D, causal, masked, scale):
    B = 2
    qkv = _qkv(B, S, H + 2 * HKV, D)
    cs, sn = _tables(D)
    pos = _positions(B * S)
    mask = None
    if masked:
        mask = torch.zeros(B, S, device="cuda")
        mask[1, S // 2 + 1:] = float("-inf")
    want_qkv = ops.rope_qk_(qkv.clone(), cs, sn, pos, H + HKV)
    want = ops.attn_fwd(want_qkv[:, :, :H], want_qkv[:, :, H: H + HKV],
                        want_qkv[:, :, H + HKV:], mask=mask, causal=causal,
                        scale=scale)
    own = qkv.clone()
    out = ops.rope_attn_(own, cs, sn, pos, H, HKV, mask=mask, causal=causal,
                         scale=scale)
    assert torch.equal(own[:, :, H:], want_qkv[:, :, H:])
    _same(out, want)


@pytest.mark.parametrize("lens", [[1], [128, 1, 127], [300, 64, 129]])
@pytest.mark.parametrize("H,HKV,D", [(2, 2, 64), (4, 2, 128)])
def test_packed(lens, H, HKV, D):
    T = sum(lens) + 3  # rows that no sequence holds
    cu = torch.tensor([0] + lens, device="cuda").cumsum(0).int()
    qkv = _qkv(T, H + 2 * HKV, D)
    cs, sn = _tables(D)
    pos = _positions(T)
    want_qkv = ops.rope_qk_(qkv.clone(), cs, sn, pos, H + HKV)
    want = ops.attn_varlen(want_qkv[:, :H], want_qkv[:, H: H + HKV],
                           want_qkv[:, H + HKV:], cu)
    own = qkv.clone()
    out = ops.rope_attn_varlen_(own, cs, sn, pos, H, HKV, cu)
    assert torch.equal(own[:, H:], want_qkv[:, H:])
    _same(out, want)


@pytest.mark.parametrize("D", [64, 96])
def test_general(D):
    """Rows that are no multiples of 16 bytes apart, heads of other sizes."""
    B, S, H, HKV = 2, 40, 4, 2
    flat = _qkv(B * S * (H + 2 * HKV) * D + 1)
    cs, sn = _tables(D)
    pos = _positions(B * S)
    for at in (0, 1):
        qkv = flat[at: at + flat.numel() - 1].view(B, S, H + 2 * HKV, D)
        want_qkv = ops.rope_apply(qkv, cs, sn, pos, rope_heads=H + HKV)
        want = ops.attn_fwd(want_qkv[:, :, :H].clone(),
                            want_qkv[:, :, H: H + HKV].clone(),
                            want_qkv[:, :, H + HKV:].clone(), causal=True)
        keep = flat.clone()
        out = ops.rope_attn_(qkv, cs, sn, pos, H, HKV, causal=True)
        flat = keep
        _same(out, want)


@pytest.mark.parametrize("S", [32, 300, 1000])
@pytest.mark.parametrize("H,HKV,D", [(6, 6, 64), (8, 2, 128)])
def test_bits(S, H, HKV, D):
    """The queries that attention rotates are those of the launch that rotates keys,
    bit for bit: no output depends on which of them a call took."""
    qkv = _qkv(3, S, H + 2 * HKV, D)
    cs, sn = _tables(D)
    pos = _positions(3 * S)
    turned = ops.rope_qk_(qkv.clone(), cs, sn, pos, H + HKV)
    want = ops.attn_fwd(turned[:, :, :H], turned[:, :, H: H + HKV],
                        turned[:, :, H + HKV:], causal=True)
    assert torch.equal(want, ops.rope_attn_(qkv.clone(), cs, sn, pos, H, HKV,
                                            causal=True))
    cu = torch.tensor([0, S, 3 * S], device="cuda", dtype=torch.int32)
    flat = turned.view(3 * S, H + 2 * HKV, D)
    want = ops.attn_varlen(flat[:, :H], flat[:, H: H + HKV],
                           flat[:, H + HKV:], cu)
    assert torch.equal(want, ops.rope_attn_varlen_(
        qkv.view(flat.shape).clone(), cs, sn, pos, H, HKV, cu))
