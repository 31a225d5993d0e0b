"""What precedes and follows an encoder's layers: embeddings with their norm,
key masks, rotation in place, pooled means."""

import pytest
import torch

from distllm_amd import ops
from distllm_amd.models import build_model
from distllm_amd.ops import torch_ref

pytestmark = pytest.mark.gpu


def _some(device, *s, seed=0):
    g = torch.Generator(device=device).manual_seed(seed)
    return torch.randn(*s, device=device, generator=g).to(torch.bfloat16)


@pytest.mark.parametrize("H", [8, 512, 520, 768, 1280, 8192])
@pytest.mark.parametrize("own", [False, True])
def test_embed_layer_norm(device, H, own):
    word, pos, row = (_some(device, n, H, seed=n) for n in (50, 12, 1))
    w, b = _some(device, H, seed=1), _some(device, H, seed=2)
    ids = torch.randint(-50, 50, (3, 11), device=device)  # negative: from
    at = torch.randint(0, 12, (3, 11), device=device) if own else None
    got = ops.embed_layer_norm(ids, at, word, pos, row[0], w, b, 1e-5)
    p = pos[:11][None] if at is None else pos[at]
    want = torch.nn.functional.layer_norm(
        word[ids].float() + p.float() + row[0].float(), (H,), w.float(),
        b.float(), 1e-5)
    torch.testing.assert_close(got.float(), want, atol=1e-2, rtol=8e-3)


@pytest.mark.parametrize("strided", range(3))
def test_embed_layer_norm_of_strided_tables(device, strided):
    """Tables that are views of others."""
    args = [_some(device, 50, 64), _some(device, 12, 64, seed=1),
            *(_some(device, 64, seed=n) for n in (2, 3, 4))]
    ids = torch.randint(0, 50, (3, 11), device=device)
    want = ops.embed_layer_norm(ids, None, *args, 1e-5)
    t = args[strided]
    args[strided] = torch.stack([t, t], -1)[..., 0]
    got = ops.embed_layer_norm(ids, None, *args, 1e-5)
    # here sums are rounded to bf16 ahead of the norm
    torch.testing.assert_close(got, want, atol=4e-2, rtol=2e-2)


@pytest.mark.parametrize("dtype", [torch.bool, torch.int8, torch.uint8,
                                   torch.int16, torch.int32, torch.int64,
                                   torch.float32])
def test_key_bias(device, dtype):
    m = (torch.arange(600, device=device).view(2, 300) % 3).to(dtype)
    want = torch.where(m.bool(), 0.0, float("-inf"))
    assert torch.equal(ops.key_bias(m), want)
    assert torch.equal(ops.key_bias(m.t()), want.t())


@pytest.mark.parametrize("D", [16, 64, 128])
@pytest.mark.parametrize("Hx,heads", [(1, 1), (3, 2), (9, 9), (48, 40),
                                      (20, 0)])
@pytest.mark.parametrize("rows", [1, 7, 130])
def test_rope_in_place(device, rows, Hx, heads, D):
    cs, sn = ops.rope_tables(64, D, device=device)
    x = _some(device, rows, Hx, D, seed=rows)
    pos = torch.arange(rows, device=device, dtype=torch.int32) * 5 % 64
    want = torch_ref.rope_apply(x, cs, sn, pos, rope_heads=heads)
    if heads == 0:
        want = x.clone()
    got = ops.rope_qk_(x, cs, sn, pos, heads)
    assert got is x
    assert torch.equal(x[:, heads:], want[:, heads:])
    # one rounding of sums of two products that may cancel
    torch.testing.assert_close(x.float(), want.float(), atol=4e-3,
                               rtol=2 ** -7)


@pytest.mark.parametrize("normalize", [False, True])
@pytest.mark.parametrize("H", [8, 320, 768, 1280, 4096])
@pytest.mark.parametrize("R,S", [(1, 1), (1, 24), (3, 33), (2, 700),
                                 (600, 40)])
def test_mean_pool(device, R, S, H, normalize):
    x = _some(device, R, S, H, seed=S)
    mask = torch.zeros(R, S, device=device, dtype=torch.int32)
    for r in range(R):
        mask[r, : max(1, S - 5 * r % S)] = 1
    got = ops.mean_pool(x, mask, normalize)
    want = torch_ref.mean_pool(x.double(), mask, False).double()
    if normalize:
        want = torch.nn.functional.normalize(want, dim=-1)
    # fp32 sums of up to 700 numbers of unit size
    torch.testing.assert_close(got.double(), want, atol=2e-6, rtol=2e-5)


@pytest.mark.parametrize("R,S", [(1, 9), (3, 40), (2, 300), (600, 24)])
def test_mean_pool_is_rounded_once(device, R, S):
    """Sums of small whole numbers have no error, so a mean is their quotient
    to the last bit."""
    x = torch.randint(-99, 100, (R, S, 320), device=device).to(torch.bfloat16)
    mask = torch.ones(R, S, device=device, dtype=torch.int32)
    total = x[:, 1:-1].double().sum(1)
    assert torch.equal(ops.mean_pool(x, mask), (total / (S - 2)).float())


@pytest.mark.parametrize("H", [8, 520, 768, 2048, 2056, 8192])
@pytest.mark.parametrize("dtype", [torch.bool, torch.int8, torch.int32,
                                   torch.int64])
def test_embed_with_bias(device, H, dtype):
    """As the two ops on their own, bit for bit."""
    g = torch.Generator(device=device).manual_seed(H)
    tables = [torch.randn(*n, H, device=device, generator=g).bfloat16()
              for n in ((50,), (40,), (), (), ())]
    ids = torch.randint(0, 50, (3, 37), device=device, generator=g)
    mask = torch.randint(0, 3, (37, 3), device=device, generator=g).t()
    mask = (mask * 2 ** 33 if dtype == torch.int64 else mask).to(dtype)
    x, bias = ops.embed_with_bias(ids, None, mask, *tables, 1e-5)
    assert torch.equal(x, ops.embed_layer_norm(ids, None, *tables, 1e-5))
    assert torch.equal(bias, ops.key_bias(mask)) and bias.is_contiguous()


@pytest.mark.parametrize("name", ["embed_layer_norm", "key_bias"])
def test_a_replaced_end_sees_its_call(device, monkeypatch, name):
    model = build_model("bert-tiny", device=device, dtype=torch.bfloat16)
    ids = torch.randint(1, 50, (2, 9), device=device)
    mask = torch.ones_like(ids)
    want, seen, own = model(ids, mask), [], getattr(ops, name)
    monkeypatch.setattr(ops, name, lambda *a: seen.append(name) or own(*a))
    assert torch.equal(model(ids, mask), want) and seen == [name]


def test_rows_without_numbers(device):
    """Nothing is read for them, and the mask is as ever."""
    tables = [torch.zeros(*n, 0, device=device, dtype=torch.bfloat16)
              for n in ((50,), (40,), (), (), ())]
    ids = torch.randint(0, 50, (3, 37), device=device)
    mask = torch.randint(0, 2, (3, 37), device=device)
    x, bias = ops.embed_with_bias(ids, None, mask, *tables, 1e-5)
    assert x.shape == (3, 37, 0) and torch.equal(bias, ops.key_bias(mask))
    assert ops.embed_layer_norm(ids, None, *tables, 1e-5).shape == x.shape
