"""The best rows of a corpus without the matrix of scores: edges of the tiles, rows
that f16 parts do not hold, equal scores."""
import pytest
import torch

from distllm_amd import ops
from distllm_amd.ops import _hip_ops

pytestmark = pytest.mark.gpu


def _unit(n, k, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(n, k, device="cuda", generator=g)
    return x / x.norm(dim=1, keepdim=True)


def _check(q, c, k):
    v, i = _hip_ops.score_topk(q, c, k)
    s = q.double() @ c.double().t()
    assert v.shape == i.shape == (len(q), k) and i.dtype == torch.int32
    assert all(len(set(r)) == k for r in i.tolist())
    assert (v[:, :-1] >= v[:, 1:]).all()
    # a float32 sum of K products, each rounded once or twice
    size = (q.double().abs() @ c.double().abs().t()).amax(1, keepdim=True)
    bound = size * q.shape[1] * 2 ** -23
    assert ((v - s.gather(1, i.long())).abs() <= bound).all()
    assert ((v - s.topk(k).values).abs() <= 2 * bound).all()


@pytest.mark.parametrize("Q", [1, 64, 65, 128, 129, 256, 257, 520])
@pytest.mark.parametrize("N, K, k", [(60, 32, 60), (129, 256, 1),
                                     (1000, 288, 60), (4098, 320, 10),
                                     (33000, 384, 7)])
def test_edges(device, Q, N, K, k):
    _check(_unit(Q, K, Q), _unit(N, K, N), k)


@pytest.mark.parametrize("Q", [64, 100, 256])
@pytest.mark.parametrize("form", ["large", "small", "some", "late", "zero"])
def test_ranges(device, Q, form):
    """Corpora beyond f16 parts as a whole, in a few rows, in columns that come
    late, and rows of zeros, which are within."""
    q, c = _unit(Q, 256, 1), _unit(40000, 256, 2)
    if form == "large":
        c *= 1e3
    elif form == "small":
        c *= 1e-5
    elif form == "some":
        c[7::1111] *= 1e3
        c[39999] *= 1e-6
    elif form == "late":
        c[5000:5300, 255] = 70.0
    else:
        c[100:400] = 0
    _check(q, c, 10)


@pytest.mark.parametrize("Q, N, K", [(100, 30001, 288), (256, 40000, 256),
                                     (520, 20000, 320)])
@pytest.mark.parametrize("small", [6e-3, 1e-3, 1e-6, 1e-9, 1e-11, 1e-13])
@pytest.mark.parametrize("form", ["corpus", "queries", "some"])
def test_wide_range(device, Q, N, K, small, form):
    """A number in every row of the corpus beside which the others, which decide, are
    small, and which the queries do not weigh; the other way round; queries that do
    among those that do not. (Beside 6e-3 it is the tenth best score that shows it,
    from 1e-3 down a sample.)"""
    q, c = _unit(Q, K, 1), _unit(N, K, 2)
    wide, other = (q, c) if form == "queries" else (c, q)
    wide *= small
    wide[:, 0] = 1
    if form == "some":
        other[::3, 0] = 0
    else:
        other[:, 0] = 0
    _check(q, c, 10)


@pytest.mark.parametrize("Q", [64, 70, 200])
def test_equal_scores_by_place(device, Q):
    """Rows that occur several times; a query of zeros, for which more groups are
    equal than the buffer holds."""
    q, c = _unit(Q, 256, 3), _unit(20000, 256, 4)
    c[[300, 4000, 17, 19999, 4003]] = q[5]
    q[9] = 0
    _, i = _hip_ops.score_topk(q, c, 20)
    assert i[5, :5].tolist() == [17, 300, 4000, 4003, 19999]
    assert i[9].tolist() == list(range(20))


@pytest.mark.parametrize("Q", [70, 200])
def test_not_finite(device, Q):
    """Infinities, NaN and numbers beyond f16 as in float32 sums."""
    q, c = _unit(Q, 256, 5), _unit(3000, 256, 6)
    # 256 numbers of a unit vector sum to 16 at most: no order of the products
    # with the large row leaves float32, which 3e38 would in some
    c[100, 5], c[2000, 7], c[2500] = float("inf"), float("nan"), 1e37
    q[7, 7] = float("-inf")
    v, i = _hip_ops.score_topk(q, c, 10)
    want, at = ops.topk(_hip_ops.score(q, c), 10)
    assert torch.equal(v.isnan(), want.isnan())
    assert torch.equal(i, at)
    torch.testing.assert_close(v, want, equal_nan=True, rtol=1e-5, atol=1e-6)


def test_refusals(device):
    q, c = _unit(40, 64, 7), _unit(50, 64, 8)
    for k in (0, 51, 61):
        with pytest.raises(RuntimeError):
            _hip_ops.score_topk(q, c, k)
    v, i = ops.score_topk(q, c, 55)
    assert v.shape == (40, 55) and (i[:, 50:] == -1).all()


def test_place_of_a_query(device):
    """What a query finds does not depend on its place in the batch, with rows beyond
    f16 parts in one share of the corpus (every tile of queries looks at all of it)."""
    q, c = _unit(256, 256, 9), _unit(40000, 256, 10)
    c[:10000] *= 1e3
    v, i = _hip_ops.score_topk(q.repeat(4, 1), c, 10)
    for at in (256, 512, 768):
        assert torch.equal(v[at: at + 256], v[:256])
        assert torch.equal(i[at: at + 256], i[:256])
    _check(q, c, 10)


@pytest.mark.parametrize("Q", [65, 128, 256, 520])
@pytest.mark.parametrize("N, K", [(70001, 288), (66000, 352), (90000, 256)])
def test_runs_of_tiles(device, Q, N, K):
    """Workgroups of several tiles: odd and even numbers of steps over their edges, the
    last tile whole and not, a tile in the middle that is made by bf16 parts."""
    q, c = _unit(Q, K, Q), _unit(N, K, K)
    _check(q, c, 12)
    c[N // 2: N // 2 + 3] *= 1e4
    _check(q, c, 12)


def test_captured(device):
    """Replays of one graph over queries that f16 parts do for, that they lose too much
    of, and back: which launches do the work is decided on the device."""
    c = _unit(30000, 256, 11)
    c[:, 0] = 1
    c[:, 1:] *= 6e-3
    plain, blind = _unit(100, 256, 12), _unit(100, 256, 13)
    blind[:, 0] = 0
    q = plain.clone()
    _hip_ops.score_topk(q, c, 10)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        v, i = _hip_ops.score_topk(q, c, 10)
    for now in (plain, blind, plain, blind):
        q.copy_(now)
        graph.replay()
        got = v.clone(), i.clone()
        want = _hip_ops.score_topk(now, c, 10)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
        _check(now, c, 10)
        torch.cuda.synchronize()
