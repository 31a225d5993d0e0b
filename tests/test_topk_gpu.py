"""Top-k at the edges of its chunks, with piled-up and equal scores."""

import pytest
import torch

from distllm_amd import ops

pytestmark = pytest.mark.gpu


def _check(scores, k):
    v, i = ops.topk(scores, k)
    n = min(k, scores.shape[1])
    want = scores.sort(dim=1, descending=True).values[:, :n]
    assert v.shape == i.shape == (scores.shape[0], k)
    assert torch.equal(v[:, :n], want)
    # every index once, and of the score it stands beside
    assert torch.equal(scores.gather(1, i[:, :n].long()), want)
    assert all(len(set(r)) == n for r in i[:, :n].tolist())
    assert (i[:, n:] == -1).all() and torch.isinf(v[:, n:]).all()


@pytest.mark.parametrize("k", [1, 5, 256, 257, 1000])
@pytest.mark.parametrize("N", [1, 4, 255, 257, 8191, 8192, 8193, 70001])
def test_sizes(device, N, k):
    g = torch.Generator(device=device).manual_seed(N + k)
    _check(torch.randn(3, N, device=device, generator=g), k)


@pytest.mark.parametrize("k", [59, 60, 61, 64, 65, 128, 129, 200, 201])
@pytest.mark.parametrize("Q, N", [(3, 300), (3, 9000), (512, 300),
                                  (513, 300), (513, 3999), (513, 4000)])
def test_rule(device, Q, N, k):
    """Both sides of where the form changes."""
    g = torch.Generator(device=device).manual_seed(N + k)
    _check(torch.randn(Q, N, device=device, generator=g), k)


def test_refusals(device):
    s = torch.randn(2, 20000, device=device)
    for k, chunk in ((257, 8192), (0, 8192), (5, 8193), (5, 0)):
        with pytest.raises(RuntimeError):
            ops._hip_ops.topk_chunked(s, None, k, chunk, True)


@pytest.mark.parametrize("k", [1, 10, 256])
def test_few_threads_have_the_large_scores(device, k):
    """All large scores at places of one residue mod 256: far more than the
    buffer of candidates reach the first bound."""
    s = torch.rand(2, 20000, device=device)
    s[:, 3::256] += 10
    s[:, :8192] = torch.linspace(1, 2, 8192, device=device)
    _check(s, k)
    _check(s.flip(1).contiguous(), k)


@pytest.mark.parametrize("k", [1, 7, 200])
def test_equal_scores(device, k):
    s = torch.zeros(2, 30000, device=device)
    _check(s, k)
    s[:, 12345:12350] = 1.0
    _check(s, k)
    s[1] = float("-inf")
    s[1, 17] = torch.finfo(torch.float32).min
    v, i = ops.topk(s, k)
    assert i[1, 0] == 17 and torch.isinf(v[1, 1:]).all()


def test_equal_scores_by_place(device):
    """Among a moderate number of equals the first places win."""
    s = torch.randn(1, 8000, device=device)
    s[0, 100::500] = 9.0
    _, i = ops.topk(s, 5)
    assert i[0].tolist() == [100, 600, 1100, 1600, 2100]


@pytest.mark.parametrize("k", [1, 7, 60, 61, 100, 200])
@pytest.mark.parametrize("N", [5000, 8192, 30000])
def test_many_equal_scores_by_place(device, N, k):
    """Also among more equals than the buffer of candidates holds, with and
    without larger scores ahead of them; the same on every call."""
    s = torch.zeros(3, N, device=device)
    s[1, N // 2] = s[1, 11] = 1.0
    s[2, ::2] = -1.0
    want = torch.stack([
        torch.arange(k), torch.tensor(([11, N // 2] + [
            i for i in range(k + 2) if i != 11])[:k]),
        torch.arange(k) * 2 + 1])
    for _ in range(3):
        _, i = ops.topk(s, k)
        assert torch.equal(i.cpu().long(), want)


def _lists(v, i):
    v, i = v.cpu(), i.cpu()
    keep = [row >= 0 for row in i]
    return ([s[k].tolist() for s, k in zip(v, keep)],
            [x[k].tolist() for x, k in zip(i, keep)])


@pytest.mark.parametrize("Q,k", [(0, 3), (1, 0), (1, 5), (256, 10), (3, 1000)])
@pytest.mark.parametrize("form", ["topk", "apart", "swapped", "strided"])
def test_found_lists(device, Q, k, form):
    """However scores and indices lie, with entries that are none."""
    g = torch.Generator(device=device).manual_seed(Q + k)
    both = torch.empty(2, Q, k, dtype=torch.int32, device=device)
    if form == "strided":
        both = torch.empty(2, Q, 2 * k, dtype=torch.int32,
                           device=device)[:, :, ::2]
    v, i = both[0].view(torch.float32), both[1]
    if form == "apart":
        i = torch.empty_like(i)
    if form == "swapped":
        v, i = both[1].view(torch.float32), both[0]
    v.copy_(torch.randn(Q, k, device=device, generator=g))
    i.copy_(torch.randint(-2, 9, (Q, k), device=device, generator=g))
    if Q > 1:
        i[0] = -1
        i[1] = 7
        v[1, 0] = float("inf")
        v[1, -1] = float("-inf")
    want = _lists(v, i)
    got = ops.found_lists(v, i)
    assert got == want
    assert all(type(x) is int for row in got[1] for x in row)
    assert all(type(x) is float for row in got[0] for x in row)
    if form == "topk" and k:
        found = ops.topk(torch.randn(max(Q, 1), 5000, device=device), k)
        assert ops.found_lists(*found) == _lists(*found)
