"""The native call for few rows against the same layers one by one, at the
edges of its rule, with masks, and where it has to stand back."""

import pytest
import torch

from distllm_amd import ops
from distllm_amd.models import ModelDims, build_model

pytestmark = pytest.mark.gpu


def _model(device, H=128, heads=2, ff=256, gelu="erf", layers=3):
    torch.manual_seed(H + ff)
    m = build_model(ModelDims(
        arch="bert", vocab_size=300, hidden_size=H, num_layers=layers,
        num_heads=heads, intermediate_size=ff, max_position_embeddings=80,
        gelu=gelu), device=device)
    with torch.no_grad():
        for p in m.parameters():
            p.add_(torch.randn_like(p) * 0.05)
    return m


def _layers(m, ids, mask):
    """The general path: a hook that changes nothing turns the call off."""
    hooks = [x.register_forward_hook(lambda *a: None) for x in m.layers]
    out = m(ids, mask)
    for h in hooks:
        h.remove()
    return out


@pytest.mark.parametrize("H,heads,ff", [(128, 2, 256), (128, 1, 64),
                                        (768, 12, 3072), (192, 3, 320)])
@pytest.mark.parametrize("B,S", [(1, 1), (1, 24), (3, 21), (1, 64), (13, 5)])
def test_same_as_layers(device, B, S, H, heads, ff):
    m = _model(device, H, heads, ff, "tanh" if H == 192 else "erf")
    ids = torch.randint(0, 300, (B, S), device=device)
    mask = (torch.arange(S, device=device)[None]
            < torch.randint(1, S + 1, (B, 1), device=device)).int()
    calls = []
    real = ops._hip_ops.bert_few_rows

    class Spy:
        def __getattr__(self, n):
            return getattr(ops_mod, n)

        @staticmethod
        def bert_few_rows(*a):
            calls.append(1)
            return real(*a)

    ops_mod = ops._hip_ops
    ops._hip_ops = Spy()
    try:
        out = m(ids, mask)
    finally:
        ops._hip_ops = ops_mod
    assert bool(calls) == (B * S <= 64 and ff >= 128)
    assert torch.equal(out, _layers(m, ids, mask))


@pytest.mark.parametrize("B,S,H,heads,ff", [
    (1, 9, 768, 12, 768), (1, 25, 768, 12, 3072), (1, 32, 1024, 16, 4096),
    (1, 33, 768, 12, 3072), (2, 12, 1024, 16, 1024), (2, 16, 768, 12, 3072),
    (2, 24, 512, 8, 2048), (3, 15, 512, 8, 512), (4, 8, 384, 6, 1536),
    (24, 1, 64, 1, 128), (6, 10, 256, 4, 256), (5, 8, 832, 13, 128)])
def test_joined_launches(device, B, S, H, heads, ff):
    """Norms and attention within a product's launch: their edges of rows,
    width and texts, odd starts of texts, and a text without tokens."""
    m = _model(device, H, heads, ff, "tanh" if ff == H else "erf")
    ids = torch.randint(0, 300, (B, S), device=device)
    at = torch.arange(B, device=device)[:, None]
    mask = (torch.arange(S, device=device)[None] < (S - at * 3) % (S + 1))
    if B == 1:
        mask[:, S // 2] = False
    assert torch.equal(m(ids, mask.int()), _layers(m, ids, mask.int()))


@pytest.mark.parametrize("S", [16, 24, 25, 32])
@pytest.mark.parametrize("H,heads", [(768, 12), (832, 13), (1024, 16)])
def test_norms_on_both_sides_of_their_bound(device, S, H, heads):
    """Joined with a product up to 32 rows of 768, 24 of more."""
    m = _model(device, H, heads, 256)
    ids = torch.randint(0, 300, (1, S), device=device)
    mask = torch.ones_like(ids)
    assert torch.equal(m(ids, mask), _layers(m, ids, mask))


def test_stands_back(device):
    m = _model(device)
    ids = torch.randint(0, 300, (1, 20), device=device)
    mask = torch.ones_like(ids)
    seen = []
    h = m.layers[1].register_forward_hook(lambda *a: seen.append(1))
    out = m(ids, mask)
    h.remove()
    assert seen == [1]
    assert torch.equal(out, m(ids, mask))
    m.layers[2].w1.data = m.layers[2].w1.data.t().contiguous().t()
    assert torch.allclose(out.float(), m(ids, mask).float(), atol=0.1)


def test_streams(device):
    """Calls on two streams at once keep to their own buffers."""
    m = _model(device, 768, 12, 3072)
    ids = [torch.randint(0, 300, (1, 20 + i), device=device)
           for i in range(2)]
    want = [m(i, torch.ones_like(i)) for i in ids]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in ids]
    for _ in range(5):
        got = []
        for s, i in zip(streams, ids):
            with torch.cuda.stream(s):
                got.append(m(i, torch.ones_like(i)))
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_layers_of_different_sizes(device):
    """A layer whose feed-forward is of another size than the first's."""
    m = _model(device)
    ids = torch.randint(0, 300, (1, 20), device=device)
    mask = torch.ones_like(ids)
    x = m.layers[1]
    with torch.no_grad():
        x.w1 = torch.nn.Parameter(x.w1[:192].clone())
        x.b1 = torch.nn.Parameter(x.b1[:192].clone())
        x.w2 = torch.nn.Parameter(x.w2[:, :192].contiguous())
    assert torch.equal(m(ids, mask), _layers(m, ids, mask))
