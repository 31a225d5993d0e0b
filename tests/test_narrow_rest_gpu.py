"""Questions that rows in 16 bits leave open, for rows that are nearly as good as
the best or for their numbers: only they are asked again."""
import threading

import numpy as np
import pytest
import torch

from distllm_amd import ops
from distllm_amd.ops import _hip_ops
from distllm_amd.rag.search import HipFlatIndex

pytestmark = pytest.mark.gpu


def _unit(n, k, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(n, k, device="cuda", generator=g)
    return x / x.norm(dim=1, keepdim=True)


def _found(q, c, k):
    n = ops.narrow_rows(c)
    return _hip_ops.narrow_found(q.cpu(), c, n.rows, n.up, n.error, n.norm, k,
                                 True)


def _beside(q, c, rows, noise):
    """c with questions' own vectors, nearly, in the places `rows` [some, many]."""
    g = torch.Generator(device="cuda").manual_seed(3)
    for i, at in enumerate(rows):
        c[at] = q[i] + noise * torch.randn(len(at), c.shape[1], device="cuda",
                                           generator=g)
    return c


def _check(found, q, c, k, rest, equal):
    scores, rows, left = found
    assert left == rest
    s = q.double() @ c.double().t()
    # a float32 sum of K products, each rounded once or twice
    bound = (q.double().abs() @ c.double().abs().t()).max() * (
        c.shape[1] * 2 ** -23)
    best = s.topk(k).values
    for i in range(len(q)):
        if i in rest:
            assert scores[i] == rows[i] == []
            continue
        assert len(set(rows[i])) == k
        at = torch.tensor(rows[i], device="cuda")
        v = torch.tensor(scores[i], device="cuda", dtype=torch.float64)
        assert (v[:-1] >= v[1:]).all()
        assert ((v - s[i, at]).abs() <= bound).all()
        assert ((v - best[i]).abs() <= 2 * bound).all()
    for i, at in enumerate(equal):  # by place
        assert rows[i] == sorted(at.tolist())[:k]


@pytest.mark.parametrize("k", [1, 10, 60])
@pytest.mark.parametrize("noise", [0, 1e-6])
@pytest.mark.parametrize("Q, N, K, many, some, every", [
    (1, 40000, 64, 1100, 1, 1),      # more groups than are scored at once
    (3, 40000, 96, 4500, 3, 1),      # than have room in a list
    (1, 250000, 32, 5000, 1, 50),    # in more spans than are looked into
    (2, 9001, 256, 1100, 1, 7),      # beside a question that is answered
    (40, 40003, 64, 900, 5, 8),      # of a batch
    (32, 70000, 64, 1060, 32, 1),    # as many as are asked again
    (200, 70001, 128, 1200, 4, 1),
    (4100, 40000, 1024, 1100, 1, 1)])  # whose answer is copied
def test_near_rows(device, k, noise, Q, N, K, many, some, every):
    q, c = _unit(Q, K, 1), _unit(N, K, 2)
    at = (torch.arange(many)[None] * every
          + torch.arange(some)[:, None] * (N // some) + N // 7) % N
    at = at.cuda()
    c = _beside(q, c, at, noise)
    assert _hip_ops.narrow_found(
        q.cpu(), c, *(lambda n: (n.rows, n.up, n.error, n.norm))(
            ops.narrow_rows(c)), k) is None
    _check(_found(q, c, k), q, c, k, [], at if noise == 0 else [])


@pytest.mark.parametrize("Q, N, many, some, rest", [
    (1, 40000, 24000, 1, [0]), (50, 70000, 1040, 33, list(range(33))),
    (5, 3000, 1600, 1, [0])])
def test_rows_of_which_the_corpus_is_read_in_less(device, Q, N, many, some,
                                                  rest):
    q, c = _unit(Q, 64, 1), _unit(N, 64, 2)
    at = (torch.arange(many)[None] + torch.arange(some)[:, None] * (N // some)
          ) % N
    c = _beside(q, c, at.cuda(), 0)
    _check(_found(q, c, 10), q, c, 10, rest, [])


@pytest.mark.parametrize("Q", [7, 130, 4097])
def test_numbers(device, Q):
    """Infinite, NaN and tiny ones are left; zeros have all rows alike. Of 4097
    the answer is copied."""
    q, c = _unit(Q, 1024, 1), _unit(900, 1024, 2)
    q[0, 5], q[1, 95], q[3] = float("inf"), float("nan"), q[3] * 1e-37
    q[2] = q[Q - 1] = 0
    q[2, 7] = -0.0
    scores, rows, left = _found(q, c, 9)
    assert left == [0, 1, 3]
    for i in (2, Q - 1):
        assert rows[i] == list(range(9)) and scores[i] == [0.0] * 9
        v, x = ops.score_topk(q[i:i + 1], c, 9)
        assert rows[i] == x[0].tolist() and scores[i] == v[0].tolist()
    sure = [i for i in range(Q) if i not in (0, 1, 2, 3, Q - 1)]
    want = _found(q[sure].contiguous(), c, 9)
    assert [rows[i] for i in sure] == want[1]
    assert [scores[i] for i in sure] == want[0]


def _index(tmp_path, c):
    from datasets import Dataset

    Dataset.from_dict({"text": ["a"]}).save_to_disk(str(tmp_path / "d"))
    np.savez(tmp_path / "i.npz", embeddings=c.cpu().numpy())
    return HipFlatIndex(tmp_path / "d", tmp_path / "i.npz")


def test_index_asks_again_for_what_is_left(device, tmp_path, monkeypatch):
    q, c = _unit(20, 128, 1), _unit(5000, 128, 2)
    c[1000:4000] = q[4]  # more than the share of the corpus that is looked at
    q[9] *= 1e-30
    index, seen = _index(tmp_path, c), []
    own = ops.score_topk
    monkeypatch.setattr(ops, "score_topk",
                        lambda x, *a: seen.append(x) or own(x, *a))
    found = index.search(q.cpu().numpy(), 6)
    assert len(seen) == 1 and torch.equal(seen[0], q[[4, 9]])
    s = q.double() @ c.double().t()
    assert found.total_indices[4] == list(range(1000, 1006))
    for i in range(20):
        if i != 4:
            assert found.total_indices[i] == s[i].topk(6).indices.tolist()
        np.testing.assert_allclose(
            found.total_scores[i], s[i].topk(6).values.cpu(), rtol=1e-5,
            atol=0 if i == 9 else 1e-6)


def test_streams_and_threads(device, tmp_path):
    """Searches of one index by threads, each on a stream of its own, some with
    questions that are asked again."""
    c = _unit(30000, 128, 2)
    c[1000:2500] = c[0]
    index = _index(tmp_path, c)
    q = [_unit(n, 128, n) for n in (1, 3, 40, 140)]
    q[2][3] = q[1][0] = c[0]
    want = [index.search(x.cpu().numpy(), 7) for x in q]
    errors = []

    def work(x, w):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(20):
                    assert index.search(x.cpu().numpy(), 7) == w
        except BaseException as e:
            errors.append(e)

    threads = [threading.Thread(target=work, args=a) for a in zip(q, want)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors


def test_pinned_memory(device):
    assert _hip_ops.pinned(64).is_pinned()
