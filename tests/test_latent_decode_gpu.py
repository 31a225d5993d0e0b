"""Attention of single-token rows over paged latents at the edges of its
tiles, shares and head groups, against float64."""
import math

import pytest
import torch

from distllm_amd import ops

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _exact(q, cache, bt, ctx, window, scale, rank):
    """Output, and the weighted sum of the values' magnitudes."""
    out = torch.zeros(q.shape[0], q.shape[1], rank, dtype=torch.float64)
    size = torch.zeros_like(out)
    q, cache = q.cpu().double(), cache.cpu().double()
    for r, L in enumerate(ctx):
        if L == 0:
            continue
        c = cache[bt[r].long()].flatten(0, 1)[max(0, L - window):L]
        p = torch.softmax(q[r] @ c.t() * scale, -1)
        out[r], size[r] = p @ c[:, :rank], p @ c[:, :rank].abs()
    return out, size


@pytest.mark.parametrize("H", [1, 16, 17, 40])
@pytest.mark.parametrize("rank, rot", [(64, 0), (192, 64), (256, 0),
                                       (384, 0), (512, 0), (512, 64)])
def test_tiles_and_shares(device, rank, rot, H):
    """Contexts round the 64 keys of a tile, past the 64 tiles whose pages
    are looked up at once, none; numbers behind the last key that are not
    finite; any number of shares."""
    ctx = [1, 63, 64, 65, 0, 700, 4097, 4300, 16]
    g = torch.Generator().manual_seed(H + rank)
    need = [-(-max(L, 1) // 16) for L in ctx]
    perm = torch.randperm(sum(need), generator=g).int() + 1
    bt = torch.zeros(len(ctx), max(need), dtype=torch.int32)
    at = 0
    for r, n in enumerate(need):
        bt[r, :n] = perm[at: at + n]
        at += n
    cache = torch.randn(at + 1, 16, rank + rot, generator=g).to(BF16)
    for r, L in enumerate(ctx):
        if L % 16:
            cache[bt[r, L // 16], L % 16:] = float("nan")
    q = torch.randn(len(ctx), H, rank + rot, generator=g).to(BF16)
    scale = 2.0 / (rank + rot) ** 0.5
    on = [t.cuda() for t in (q, cache, bt)]
    seq = torch.arange(len(ctx), dtype=torch.int32, device="cuda")
    lens = torch.tensor(ctx, dtype=torch.int32, device="cuda")
    for window in (1 << 30, 1000, 64):
        want, size = _exact(q, cache.nan_to_num(), bt, ctx, window, scale,
                            rank)
        for nsplit in (0, 1, 5, 64, 100):
            got = ops.latent_attn(on[0], on[1], on[2], seq, lens, window,
                                  scale, nsplit, rank).cpu().double()
            # weights and output are rounded to bf16, by half of the last of
            # 7 bits behind the point: 2^-8 of each; scores are off by
            # float32 sums of up to 576 products
            bound = size * (2 ** -8 + 2 ** -8 + 1e-4) + 1e-6
            assert ((got - want).abs() <= bound).all(), (window, nsplit)
            assert not got[4].any()


@pytest.mark.parametrize("H", [3, 20])
@pytest.mark.parametrize("rank, rot", [(64, 0), (192, 64), (512, 64)])
def test_window_within_the_last_page(device, rank, rot, H):
    """Windows of up to a page that start in the page of the last key: the
    pages ahead of it are not looked up, and what lies behind the last key must
    not reach the result from the rows that stand in for them."""
    ctx = [60, 52, 63, 64, 49, 15, 4090]
    width = 256
    g = torch.Generator().manual_seed(rank + H)
    bt = torch.arange(len(ctx) * width, dtype=torch.int32).view(-1, width)
    cache = torch.randn(bt.numel(), 16, rank + rot, generator=g).to(BF16)
    for r, L in enumerate(ctx):
        if L % 16:
            cache[bt[r, L // 16], L % 16:] = float("nan")
    q = torch.randn(len(ctx), H, rank + rot, generator=g).to(BF16)
    scale = 2.0 / (rank + rot) ** 0.5
    seq = torch.arange(len(ctx), dtype=torch.int32, device="cuda")
    lens = torch.tensor(ctx, dtype=torch.int32, device="cuda")
    for window in (1, 3, 8, 16, 17):
        want, size = _exact(q, cache.nan_to_num(), bt, ctx, window, scale,
                            rank)
        for nsplit in (0, 1, 3):
            got = ops.latent_attn(q.cuda(), cache.cuda(), bt.cuda(), seq,
                                  lens, window, scale, nsplit,
                                  rank).cpu().double()
            bound = size * (2 ** -7 + 1e-4) + 1e-6  # as above
            assert ((got - want).abs() <= bound).all(), (window, nsplit)


@pytest.mark.parametrize("H", [16, 40])
@pytest.mark.parametrize("rank", [64, 512])
@pytest.mark.parametrize("p", [2.0 ** -9 * 1.00390625 + 1e-6, 2 ** -9 * 1.0039])
def test_weights_keep_more_than_bf16(device, rank, H, p):
    """One large score of value -7 and thousands of the same small weight of
    value 1: rounded to bf16 each is off by up to 2^-9 to the same side, which
    is 3% of what is left of the sum."""
    L = 4096
    q = torch.zeros(1, H, rank + 64, dtype=BF16)
    q[0, :, rank: rank + 3] = torch.tensor([1.0, 2 ** -8, 2 ** -14])
    left = torch.full((L,), math.log(p), dtype=torch.float64)
    left[0] = 0.0
    score = torch.zeros_like(left)
    cache = torch.zeros(L, rank + 64, dtype=BF16)
    cache[:, :rank] = 1.0
    cache[0, :rank] = -7.0
    for i in range(3):
        unit = q[0, 0, rank + i].item()
        cache[:, rank + i] = ((left - score) / unit).to(BF16)
        score += cache[:, rank + i].double() * unit
    want = score.softmax(0) @ cache[:, 0].double()
    bt = torch.arange(L // 16, dtype=torch.int32, device="cuda")[None]
    got = ops.latent_attn(
        q.cuda(), cache.view(-1, 16, rank + 64).cuda(), bt,
        torch.zeros(1, dtype=torch.int32, device="cuda"),
        torch.tensor([L], dtype=torch.int32, device="cuda"), 1 << 30, 1.0, 1,
        rank).double().cpu()
    # bf16 of the result and 2^-18 of parts of together 1
    assert ((got - want).abs() <= abs(want) * 2 ** -8 + 2 ** -18).all()
