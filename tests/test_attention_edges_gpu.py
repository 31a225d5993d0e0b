"""Flash attention at the edges of its tiles and forms: remainders of the
128-query and 64-key blocks, additive masks that are not 0 / -inf, rows
without a visible key, negative scales, strided and unaligned inputs, packed
rows that no sequence holds."""

from __future__ import annotations

import math

import pytest
import torch

from distllm_amd import ops
from distllm_amd.ops import torch_ref

pytestmark = pytest.mark.gpu

# bf16 probabilities and outputs: 2^-8 each, and values of a few units
TOL = 2e-2


def _qkv(B, S, H, HKV, D, seed, device):
    g = torch.Generator(device=device).manual_seed(seed)
    return (torch.randn(B, S, h, D, device=device, generator=g,
                        dtype=torch.bfloat16) for h in (H, HKV, HKV))


def _close(out, q, k, v, mask, causal, scale):
    ref = torch_ref.attn_fwd(q.float(), k.float(), v.float(), mask, causal,
                             scale)
    torch.testing.assert_close(out.float(), ref.float(), atol=TOL, rtol=TOL)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("S", [1, 63, 64, 65, 127, 129, 200])
def test_tile_edges(device, S, causal, D):
    q, k, v = _qkv(2, S, 4, 2, D, S, device)
    _close(ops.attn_fwd(q, k, v, causal=causal), q, k, v, None, causal,
           1 / math.sqrt(D))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_general_masks(device, causal, D):
    """Per key: finite biases, the type's lowest value, -inf; one tile of
    keys all masked, one without a mask."""
    B, S = 3, 193
    q, k, v = _qkv(B, S, 2, 2, D, 7, device)
    mask = torch.zeros(B, S, device=device)
    mask[0, 70:100] = -1.5
    mask[1, 64:128] = -math.inf
    mask[2, 100:] = torch.finfo(torch.float32).min
    _close(ops.attn_fwd(q, k, v, mask=mask, causal=causal), q, k, v, mask,
           causal, 1 / math.sqrt(D))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("S", [193, 512, 4400])
def test_masked_ends(device, S, causal, D):
    """Last tiles that no row sees, a last key at either side of a tile's
    border, masked keys ahead and past the first 64 tiles, no masked key."""
    q, k, v = _qkv(4, S, 2, 1, D, 9, device)
    mask = torch.zeros(4, S, device=device)
    mask[0, 64:] = -math.inf
    mask[1, 65:] = torch.finfo(torch.float32).min
    mask[2, S - 100: S - 65] = -math.inf
    mask[2, S - 64:] = -math.inf
    _close(ops.attn_fwd(q, k, v, mask=mask, causal=causal), q, k, v, mask,
           causal, 1 / math.sqrt(D))


def test_rows_without_keys_are_zero(device):
    q, k, v = _qkv(2, 100, 2, 2, 64, 8, device)
    mask = torch.zeros(2, 100, device=device)
    mask[1] = -math.inf
    out = ops.attn_fwd(q, k, v, mask=mask)
    assert torch.isfinite(out[0]).all() and (out[1] == 0).all()


@pytest.mark.parametrize("scale", [-0.2, 0.0, 0.5])
def test_scales(device, scale):
    q, k, v = _qkv(1, 150, 2, 1, 64, 9, device)
    _close(ops.attn_fwd(q, k, v, causal=True, scale=scale), q, k, v, None,
           True, scale)


def test_growing_scores(device):
    """Running maxima that grow from tile to tile, by less and by more than
    what the rescaling is put off for."""
    q, k, v = _qkv(1, 320, 2, 2, 64, 10, device)
    k = k * torch.linspace(0.1, 6.0, 320, device=device)[None, :, None, None]
    k = k.to(torch.bfloat16)
    _close(ops.attn_fwd(q, k, v), q, k, v, None, False, 1 / 8.0)


@pytest.mark.parametrize("at", [0, 1, 8])
def test_unaligned_views(device, at):
    """Keys and values of a larger buffer, from element `at` on."""
    B, S, H, D = 2, 70, 2, 64
    g = torch.Generator(device=device).manual_seed(11)
    flat = torch.randn(3, B * S * H * D + 16, device=device, generator=g,
                       dtype=torch.bfloat16)
    q, k, v = (f[at: at + B * S * H * D].view(B, S, H, D) for f in flat)
    _close(ops.attn_fwd(q, k, v), q, k, v, None, False, 1 / 8.0)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("strided", [False, True])
def test_packed(device, strided, D):
    lens = [1, 64, 65, 128, 200, 3]
    T, H, HKV = sum(lens) + 37, 4, 2
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()],
                      dtype=torch.int32, device=device)
    g = torch.Generator(device=device).manual_seed(12)
    qkv = torch.randn(T, H + 2 * HKV, D, device=device, generator=g,
                      dtype=torch.bfloat16)
    q, k, v = qkv[:, :H], qkv[:, H: H + HKV], qkv[:, H + HKV:]
    if not strided:
        q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
    out = ops.attn_varlen(q, k, v, cu)
    n = int(cu[-1])
    ref = torch_ref.attn_varlen(q[:n].float(), k[:n].float(), v[:n].float(),
                                cu, 1 / math.sqrt(D))
    torch.testing.assert_close(out[:n].float(), ref.float(), atol=TOL,
                               rtol=TOL)
    assert out.is_contiguous() and (out[n:] == 0).all()
