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


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("D", [64, 128])
def test_many_workgroups(device, D, fp8):
    """As many as change the buffers, and one row less."""
    for B in (127, 128):
        lens = [(37 * b) % 150 for b in range(B)]
        k, v, table = _pages(B, 8, D, lens, 10, fp8, B, device)
        raw = [t.view(torch.uint8) if fp8 else t for t in (k, v)]
        q = torch.randn(B, 16, D, device=device).to(torch.bfloat16)
        ctx = torch.tensor(lens, dtype=torch.int32, device=device)
        out = ops.paged_attn(q, *raw, table, ctx)
        torch.testing.assert_close(
            out.float().cpu(), _want(q, k, v, table, lens, D ** -0.5), **TOL)


@pytest.mark.parametrize("asked", ["0", "1", "2", "7", "64", "1000"])
def test_shares_asked_for(device, asked, monkeypatch):
    """DISTLLM_PA_NSPLIT, for few long sequences and for many short ones."""
    monkeypatch.setenv("DISTLLM_PA_NSPLIT", asked)
    for lens, width in (([4000, 70], 300), ([20] * 40, 2)):
        B = len(lens)
        want = {"0": 300 // 32 if B == 2 else 1}.get(
            asked, min(int(asked), width, 64))
        assert ops._hip_ops.paged_attn_shares(B, 8, 2, width,
                                              False) == want
        k, v, table = _pages(B, 2, 64, lens, width, False, B, device)
        q = torch.randn(B, 8, 64, device=device).to(torch.bfloat16)
        ctx = torch.tensor(lens, dtype=torch.int32, device=device)
        out = ops.paged_attn(q, k, v, table, ctx)
        torch.testing.assert_close(out.float().cpu(),
                                   _want(q, k, v, table, lens, 0.125), **TOL)


def _two_scores(device, D, L, scores, values):
    """Pages of L keys whose scores (scale 1) are scores[i], in steps of
    2^-26, and whose values are values[i]."""
    k, v, table = _pages(1, 1, D, [L], L // 16, False, 3, device)
    q = torch.zeros(1, 1, D, device=device, dtype=torch.bfloat16)
    q[0, 0, :4] = torch.tensor([1.0, 2 ** -8, 2 ** -14, 2 ** -20])
    rows = torch.zeros(L, D, dtype=torch.float64)
    left = torch.tensor(scores, dtype=torch.float64)
    for i in range(4):
        rows[:, i] = (left / q[0, 0, i].item()).float().bfloat16().double()
        left = left - rows[:, i] * q[0, 0, i].item()
    vals = torch.tensor(values, dtype=torch.float64)[:, None].expand(L, D)
    at = table[0].long()
    k[at, 0] = rows.to(k.dtype).to(device).view(-1, 16, D)
    v[at, 0] = vals.to(v.dtype).to(device).view(-1, 16, D)
    ctx = torch.tensor([L], dtype=torch.int32, device=device)
    out = ops.paged_attn(q, k, v, table, ctx, 1.0)
    s = (rows @ q[0, 0].double().cpu())
    want = s.softmax(0) @ vals[:, 0].bfloat16().double()
    return out.double().cpu().flatten(), want


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("p", [2.0 ** -9 * 1.00390625 + 1e-6, 2 ** -9 * 1.0039])
def test_probabilities_keep_more_than_bf16(device, D, p):
    """One large score of value -1 and thousands of the same small
    probability of value 1: rounded to bf16 each is off by up to 2^-9 to the
    same side, and the sum by more than a bf16 step of what is left."""
    L = 4096
    out, want = _two_scores(device, D, L, [0.0] + [math.log(p)] * (L - 1),
                            [-7.0] + [1.0] * (L - 1))
    assert abs(want) < 0.2  # of parts of 0.5 and more
    # bf16 of the result, 2^-9; sums of 32 bits, 2^-24 of the parts (about 1)
    assert ((out - want).abs() <= abs(want) * 2 ** -8 + 2 ** -22).all()


@pytest.mark.parametrize("D", [64, 128])
def test_probabilities_in_32_bits(device, D):
    """Two probabilities that differ in their 17th bit and lower, of values 1
    and -1, beside the largest of value 0: what is left of them has 2^-24 of
    each as its error, not the 2^-18 of a sum of two bf16 numbers."""
    worst = 0.0
    for i in range(40):
        s = -0.03 - 0.02 * i
        d = 3e-5
        out, want = _two_scores(device, D, 16, [0.0, s, s - d] + [-60.0] * 13,
                                [0.0, 1.0, -1.0] + [0.0] * 13)
        worst = max(worst, ((out - want) / want).abs().max().item())
    # 2^-9 of bf16 and 4 * 2^-24 / 3e-5 of the probabilities (the exponential
    # to two units in the last place)
    assert worst <= 2 ** -9 + 4 * 2 ** -24 / 3e-5


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


@pytest.mark.parametrize("shares", ["1", "3"])
@pytest.mark.parametrize("D", [64, 128])
def test_infinite_values(device, D, shares, monkeypatch):
    """Infinite values come out as from sums of 32 bits: infinite, with their
    sign, and NaN only where both signs meet."""
    monkeypatch.setenv("DISTLLM_PA_NSPLIT", shares)
    lens = [200, 33, 16]
    k, v, table = _pages(3, 2, D, lens, 13, False, 1, device, 0.0)
    inf = float("inf")
    for b, key, col, x in ((0, 7, 3, inf), (0, 190, 5, -inf), (1, 32, 0, inf),
                           (2, 0, 9, inf), (2, 1, 9, -inf), (2, 3, 11, -inf)):
        v[table[b, key // 16], :, key % 16, col] = x
    # the largest probability is 1, whose low parts are nothing
    q = torch.randn(3, 8, D, device=device).to(torch.bfloat16) * 0.2
    ctx = torch.tensor(lens, dtype=torch.int32, device=device)
    out = ops.paged_attn(q, k, v, table, ctx).float().cpu()
    want = _want(q, k, v, table, lens, D ** -0.5)
    assert torch.equal(out.isnan(), want.isnan()) and want.isnan().any()
    torch.testing.assert_close(out, want, equal_nan=True, **TOL)


def _step(device, lens, H, HKV, D, fp8, width, slabs=0, seed=0):
    """A step's projections and pages whose new rows hold NaN."""
    k, v, table = _pages(len(lens), HKV, D, [n - 1 for n in lens], width, fp8,
                         seed, device)
    raw = [t.view(torch.uint8) if fp8 else t for t in (k, v)]
    cs, sn = ops.rope_tables(width * 16, D, device=device)
    g = torch.Generator().manual_seed(seed)
    shape = (len(lens), H + 2 * HKV, D)
    if slabs:
        qkv = torch.randn(slabs, *shape, generator=g).to(device)
        bias = torch.randn(shape[1] * D, generator=g).bfloat16().to(device)
    else:
        qkv, bias = torch.randn(*shape, generator=g).bfloat16().to(device), None
    ctx = torch.tensor(lens, dtype=torch.int32, device=device)
    return qkv, cs, sn, ctx, raw, table, bias


def _same_step(device, qkv, cs, sn, ctx, raw, table, bias):
    """In one launch as in two."""
    two = [t.clone() for t in raw]
    HKV, D = raw[0].shape[1], raw[0].shape[3]
    H = qkv.shape[-2] - 2 * HKV
    scale = D ** -0.5
    q = ops.rope_put(qkv, cs, sn, ctx, *two, table, bias)
    want = ops.paged_attn(q, *two, table, ctx, scale)
    plan = ops.step_plan(1, ctx, H, raw[0], table)[0]
    got = ops.step_attn(qkv, cs, sn, ctx, *raw, table, bias, scale, plan)
    assert not got.isnan().any()
    torch.testing.assert_close(got.float(), want.float(), **TOL)
    for a, b in zip(raw, two):
        torch.testing.assert_close(a, b, atol=0, rtol=0, equal_nan=True)
    return plan


def _shares(slots, lens, width):
    """Every tile of 32 keys once, a sequence's shares side by side; -> the
    numbers of shares and, in their order, the sizes of the first ones."""
    cut = [[] for _ in lens]
    sizes = []
    for i, (b, n, t0, t1, first, shares) in enumerate(slots[:, :6].tolist()):
        if b < 0:
            continue
        assert n == lens[b] and first + len(cut[b]) == i < first + shares
        cut[b].append((t0, t1, shares))
        if i == first:
            sizes.append(max(t1 - t0, 1))
    for n, c in zip(lens, cut):
        tiles = -(-min(n, width * 16) // 32)
        ends = [0] + [t1 for _, t1, _ in c]
        assert [t0 for t0, _, _ in c] == ends[:-1] and ends[-1] == tiles
        assert all(shares == len(c) for _, _, shares in c)
    return [len(c) for c in cut], sizes


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H,HKV", [(4, 4), (10, 2), (20, 1), (32, 8)])
@pytest.mark.parametrize("slabs", [0, 3])
def test_step(device, H, HKV, D, fp8, slabs):
    lens = [1, 2, 16, 17, 31, 32, 33, 127, 128, 129, 257, 320]
    _same_step(device, *_step(device, lens, H, HKV, D, fp8, 20, slabs))


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("shares", ["", "2", "7", "64"])
@pytest.mark.parametrize("lens,width,H,HKV", [
    ([4800], 300, 32, 8), ([33], 300, 8, 2), ([1, 1600, 777], 100, 20, 1)])
def test_step_shares(device, lens, width, H, HKV, shares, fp8, monkeypatch):
    """Shares joined by the last of them, those without keys among them."""
    if shares:
        monkeypatch.setenv("DISTLLM_PA_NSPLIT", shares)
    args = _step(device, lens, H, HKV, 128, fp8, width)
    slots, zeros = _same_step(device, *args)
    n, _ = _shares(slots, lens, width)
    assert not shares or n == [int(shares)] * len(lens)
    want = [k if k > 1 else 0 for k in n]
    assert zeros.view(len(lens), -1).tolist() == [
        [k] * (zeros.numel() // len(lens)) for k in want]


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("HKV,groups", [(8, 8), (1, 2), (32, 32)])
@pytest.mark.parametrize("lens", [
    [1], [8000], [0, 33], [300] * 20, list(range(1, 2048, 66)),
    [200 + 56 * (7 * i % 33) for i in range(33)], [4096] + [16] * 63,
    [3 * i for i in range(300)], [40] * 1025])
def test_step_plan(device, lens, HKV, groups, fp8):
    """The cut of the lengths that a decode step's attention goes by, at and
    around as many sequences as fill the CUs and as many as are sorted."""
    B, width = len(lens), 256
    H = 20 if HKV == 1 else 32
    pages = torch.empty(2, HKV, 16, 128, device=device,
                        dtype=torch.uint8 if fp8 else torch.bfloat16)
    table = torch.zeros(B, width, dtype=torch.int32, device=device)
    ctx = torch.tensor(lens, dtype=torch.int32, device=device)
    plan = ops.step_plan(3, ctx, H, pages, table)
    assert len(plan) == 3 and all(not row.any() for _, row in plan)
    assert plan[0][1].numel() == B * groups
    n, sizes = _shares(plan[0][0], lens, width)
    full = (512 if fp8 else 256) // groups
    if B <= 1024:
        assert sizes == sorted(sizes, reverse=True)
        assert max(n) <= 32 and sum(n) <= max(full, B + full * 2 // 3)
        for k, x in zip(n, lens):  # four tiles, but for what halving leaves
            assert k == 1 or -(-min(x, width * 16) // 32) > 4 * (k - 1)
    if lens == [8000] and groups == 8:
        assert n == [32]


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("H,HKV,D", [(32, 8, 128), (20, 1, 64)])
@pytest.mark.parametrize("slabs", [0, 3])
def test_step_rows_of_one_sequence(device, H, HKV, D, fp8, slabs):
    """Tokens of one sequence that follow each other, in any order, over the
    edge of a page and in a share of their own; and two sequences that have but
    their first page in common."""
    lens = [33, 31, 20, 34, 2001, 32, 2000, 40, 25]
    qkv, cs, sn, ctx, raw, table, bias = _step(device, lens, H, HKV, D, fp8,
                                               128, slabs)
    table[[0, 3, 5]] = table[1].clone()
    table[4] = table[6].clone()
    table[8, 0] = table[7, 0]
    slots, _ = _same_step(device, qkv, cs, sn, ctx, raw, table, bias)
    assert slots[:9, 6].tolist() == [1, 0, 0, 1, 1, 1, 0, 0, 0]


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("B,H,HKV", [(64, 32, 8), (65, 32, 8), (128, 32, 8),
                                     (33, 32, 32)])
def test_step_of_many_sequences(device, B, H, HKV, fp8):
    """From 513 groups of heads on bf16 tiles have one place in a wave's ring;
    lengths of a token to several tiles a wave, and rows without any."""
    lens = [(1, 17, 32, 0, 33, 150, 300, 600)[i % 8] for i in range(B)]
    qkv, cs, sn, ctx, raw, table, _ = _step(device, lens, H, HKV, 128, fp8, 38)
    scale, two = 128 ** -0.5, [t.clone() for t in raw]
    plan = ops.step_plan(1, ctx, H, raw[0], table)[0]
    got = ops.step_attn(qkv, cs, sn, ctx, *raw, table, None, scale, plan)
    has = ctx > 0
    assert not got[~has].any()
    some = [t[has].contiguous() for t in (qkv, ctx, table)]
    q = ops.rope_put(some[0], cs, sn, some[1], *two, some[2])
    want = ops.paged_attn(q, *two, some[2], some[1], scale)
    assert not want.isnan().any()
    torch.testing.assert_close(got[has].float(), want.float(), **TOL)
    for a, b in zip(raw, two):
        torch.testing.assert_close(a, b, atol=0, rtol=0, equal_nan=True)


@pytest.mark.parametrize("B", [1, 5, 70, 1030])
def test_plan_finds_rows_of_one_sequence(device, B):
    g = torch.Generator().manual_seed(B)
    ctx = torch.randint(0, 70, (B,), generator=g).int()
    table = torch.randint(0, 2 * B, (B, 4), generator=g).int()
    pos = ctx.long() - 1
    page = pos.clamp(min=0) // 16
    ok = (pos >= 0) & (page < 4)
    at = page.clamp(max=3)
    same = table[:, at] == table[torch.arange(B), at]  # [row, writer]
    want = (same & ok & (pos < pos[:, None])).fill_diagonal_(False).any(1)
    pages = torch.empty(2, 8, 16, 128, device=device, dtype=torch.bfloat16)
    slots, _ = ops.step_plan(1, ctx.to(device), 32, pages,
                             table.to(device))[0]
    assert torch.equal(slots[:B, 6].cpu().bool(), want)
    assert B == 1 or want.any()


def test_step_unaligned_pages(device):
    args = list(_step(device, [50, 300], 8, 2, 64, False, 20))
    odd = []
    for t in args[4]:
        flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=device)
        flat[1:] = t.reshape(-1)
        odd.append(flat[1:].view(t.shape))
    args[4] = odd
    _same_step(device, *args)


def test_step_in_a_graph(device):
    """Replayed, with other work between, as run."""
    qkv, cs, sn, ctx, raw, table, _ = _step(device, [2000, 1, 640], 32, 8, 128,
                                            False, 128)

    def run():
        plan = ops.step_plan(2, ctx, 32, raw[0], table)
        return [ops.step_attn(qkv * f, cs, sn, ctx, *raw, table, None, 0.1,
                              plan[i]) for i, f in enumerate((1.0, 0.5))]

    want = [t.clone() for t in run()]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = run()
    for _ in range(4):
        for t in got:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        run()


@pytest.mark.parametrize("shape,dtype,step", [
    ((128, 64), torch.uint8, 1), ((136, 64), torch.bfloat16, 1),
    ((4099, 2048), torch.bfloat16, 1), ((127, 64), torch.bfloat16, 1),
    ((512, 96), torch.uint8, 1), ((512, 128), torch.bfloat16, 2),
    ((40000, 1024), torch.bfloat16, 1)])
def test_step_fetches_ahead(device, shape, dtype, step):
    """Weights that come to the caches beside the attention change nothing,
    also where their rows or pieces do not divide, and past the most."""
    qkv, cs, sn, ctx, raw, table, _ = _step(device, [70, 1, 33], 32, 8, 128,
                                            False, 8)
    w = torch.ones(shape, device=device).to(dtype)[:, ::step]
    outs = []
    for ahead in (None, w):
        plan = ops.step_plan(1, ctx, 32, raw[0], table)[0]
        outs.append(ops.step_attn(qkv, cs, sn, ctx, *raw, table, None, 0.1,
                                  plan, ahead))
    assert torch.equal(*outs)
    assert bool((w == 1).all())


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("lens", [[1], [5, 0, 2], [1] * 8])
@pytest.mark.parametrize("shape,dtype", [
    ((128, 64), torch.uint8),     # eight runs of one piece, the fewest
    ((213, 64), torch.uint8),     # thirteen, and rows that are no run
    ((136, 64), torch.bfloat16), ((400, 192), torch.bfloat16),
    ((4099, 2048), torch.bfloat16)])
def test_step_fetches_ahead_of_short_contexts(device, lens, shape, dtype, fp8):
    """Where the pages are less than the weights, so that these are fetched."""
    qkv, cs, sn, ctx, raw, table, _ = _step(device, lens, 4, 1, 64, fp8, 4)
    w = torch.ones(shape, device=device).to(dtype)
    runs = shape[0] // 16 * 16 * shape[1] * w.element_size()
    assert sum(lens) * 64 * (2 if fp8 else 4) <= runs
    outs = []
    for ahead in (None, w):
        plan = ops.step_plan(1, ctx, 4, raw[0], table)[0]
        outs.append(ops.step_attn(qkv, cs, sn, ctx, *raw, table, None, 0.1,
                                  plan, ahead))
    assert torch.equal(*outs) and not outs[0].isnan().any()
    assert bool((w == 1).all())
