"""Search by way of rows in 16 bits: edges of blocks and tiles, which queries they
cannot answer, and rows that are no longer the corpus's."""
import numpy as np
import pytest
import torch

from distllm_amd import ops
from distllm_amd.ops import _hip_ops
from distllm_amd.rag.search import HipFlatIndex

pytestmark = pytest.mark.gpu
UNSURE = -2 ** 31


def _unit(n, k, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(n, k, device="cuda", generator=g)
    return x / x.norm(dim=1, keepdim=True)


def _topk(q, c, k):
    n = ops.narrow_rows(c)
    return _hip_ops.narrow_topk(q, c, n.rows, n.up, n.error, n.norm, k)


def _check(q, c, k):
    v, i = _topk(q, c, k)
    s = q.double() @ c.double().t()
    assert v.shape == i.shape == (len(q), k) and i.dtype == torch.int32
    assert all(len(set(r)) == k for r in i.tolist())
    assert (v[:, :-1] >= v[:, 1:]).all()
    # a float32 sum of K products, each rounded once or twice
    size = (q.double().abs() @ c.double().abs().t()).amax(1, keepdim=True)
    bound = size * q.shape[1] * 2 ** -23
    assert ((v - s.gather(1, i.long())).abs() <= bound).all()
    assert ((v - s.topk(k).values).abs() <= 2 * bound).all()


@pytest.mark.parametrize("Q", [1, 3, 16, 17, 128, 129, 256, 300])
@pytest.mark.parametrize("N, K, k", [(60, 32, 60), (129, 256, 1),
                                     (1000, 288, 60), (4098, 320, 10),
                                     (33000, 384, 7), (8200, 1600, 5)])
def test_edges(device, Q, N, K, k):
    _check(_unit(Q, K, Q), _unit(N, K, N), k)


@pytest.mark.parametrize("Q", [2, 40, 200])
@pytest.mark.parametrize("up", [1e-20, 1.0, 1e15])
def test_ranges(device, Q, up):
    """Numbers far from 1, all of one sign, and rows in the order of their
    scores, so that the best lie in one place."""
    q, c = _unit(Q, 256, 1).abs() / up, -_unit(40000, 256, 2).abs() * up
    _check(q, c[(c @ q[0]).argsort()].contiguous(), 10)


@pytest.mark.parametrize("Q", [1, 16, 60, 256])
def test_equal(device, Q):
    """Equal scores go by place, as far as there is room for their rows."""
    q, c = _unit(Q, 128, 1), _unit(1200, 128, 2).repeat(5, 1)
    v, i = _topk(q, c, 12)
    s = _topk(q, c[:1200].contiguous(), 3)[1]
    want = (s[:, :, None] + 1200 * torch.arange(5, device="cuda")).flatten(1)
    assert torch.equal(i, want[:, :12].int())
    v, i = _topk(q, c[:1].repeat(3000, 1), 12)
    assert (i == UNSURE).all()


@pytest.mark.parametrize("Q", [7, 130])
def test_queries_that_are_not_answered(device, Q):
    q, c = _unit(Q, 96, 1), _unit(5000, 96, 2)
    q[0, 5], q[1, 95], q[2, 0] = float("inf"), float("nan"), -float("inf")
    q[3], q[4] = 0, q[4] * 1e-37
    v, i = _topk(q, c, 9)
    assert (i[:5] == UNSURE).all()
    assert torch.equal(i[5:], _topk(q[5:].contiguous(), c, 9)[1])
    n = ops.narrow_rows(c)
    args = c, n.rows, n.up, n.error, n.norm, 9
    assert _hip_ops.narrow_found(q.cpu(), *args) is None
    assert _hip_ops.narrow_found(q[5:].cpu(), *args) == tuple(
        t.tolist() for t in (v[5:], i[5:]))


@pytest.mark.parametrize("Q", [4096, 4097])
def test_host_queries_pinned_or_copied(device, Q):
    """Q of 1024 numbers: 16 MB, and above it."""
    q, c = _unit(Q, 1024, 1), _unit(900, 1024, 2)
    n = ops.narrow_rows(c)
    found = _hip_ops.narrow_found(q.cpu(), c, n.rows, n.up, n.error, n.norm, 3)
    assert found == tuple(t.tolist() for t in _topk(q, c, 3))


def test_rows_of_no_use(device):
    c = _unit(500, 64, 1)
    assert ops.narrow_rows(c.double()) is None
    assert ops.narrow_rows(c[:, :63].contiguous()) is None
    assert ops.narrow_rows(c.flatten()[1:-63].view(-1, 64)) is None
    assert ops.narrow_rows(torch.zeros_like(c)) is None
    for x in (float("inf"), float("nan"), 1e6):
        d = c.clone()
        d[77, 3] = x
        assert ops.narrow_rows(d) is None
    with pytest.raises(RuntimeError):
        n = ops.narrow_rows(c)
        _hip_ops.narrow_topk(c[:3], c, n.rows[:16], n.up, n.error, n.norm, 4)


@pytest.mark.parametrize("Q", [1, 70])
def test_index(device, tmp_path, monkeypatch, Q):
    """Answers of an index: by the rows in 16 bits, and not by them when its
    corpus has been changed or replaced, or another search put in place."""
    from datasets import Dataset

    c, q = _unit(5000, 128, 1), _unit(Q, 128, 2)
    Dataset.from_dict({"text": ["a"]}).save_to_disk(str(tmp_path / "d"))
    np.savez(tmp_path / "i.npz", embeddings=c.cpu().numpy())
    index = HipFlatIndex(tmp_path / "d", tmp_path / "i.npz")
    calls = []
    own = _hip_ops.narrow_found
    monkeypatch.setattr(_hip_ops, "narrow_found",
                        lambda *a: calls.append(0) or own(*a), raising=False)

    def check(by):
        calls.clear()
        found = index.search(q.cpu().numpy(), 6)
        s = q.double() @ index.corpus.double().t()
        assert found.total_indices == s.topk(6).indices.tolist()
        np.testing.assert_allclose(found.total_scores, s.topk(6).values.cpu(),
                                   atol=1e-6)
        assert len(calls) == by

    check(1)
    index.corpus.mul_(-1)
    check(0)
    index.narrow = ops.narrow_rows(index.corpus)
    check(1)
    index.corpus = c.clone()
    check(0)
    index.narrow = ops.narrow_rows(index.corpus)
    monkeypatch.setattr(index, "_topk_exact",
                        lambda x, k: HipFlatIndex._topk_exact(index, x, k))
    check(0)
    monkeypatch.undo()

    def full(*a):
        raise torch.OutOfMemoryError("no room")

    monkeypatch.setattr(_hip_ops, "narrow_found", full, raising=False)
    check(0)
    monkeypatch.undo()
    # rows that are all the same are asked again
    index.corpus = c[:1].repeat(5000, 1)
    index.narrow = ops.narrow_rows(index.corpus)
    found = index.search(q.cpu().numpy(), 6)
    assert found.total_indices == [list(range(6))] * Q
