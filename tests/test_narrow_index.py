"""An index's rows in 16 bits beside its corpus: when they are its, on the CPU with
a stand-in for the search by them."""
from contextlib import nullcontext as _nothing

import numpy as np
import pytest
import torch
from datasets import Dataset

from distllm_amd import ops
from distllm_amd.rag.search import HipFlatIndex, HipIndexConfig


@pytest.fixture
def by_narrow(monkeypatch):
    """Searches by the rows in 16 bits, which answer nothing here."""
    calls = []

    def rows(corpus):
        return ops.NarrowRows(corpus.half(), 0, 0.0, 1.0, corpus,
                              corpus._version)

    monkeypatch.setattr(ops, "narrow_rows", rows)
    monkeypatch.setattr(ops, "found_narrow",
                        lambda *a: calls.append(a) and None)
    return calls


@pytest.fixture
def index(tmp_path, by_narrow):
    c = torch.randn(50, 8, generator=torch.Generator().manual_seed(1))
    Dataset.from_dict({"text": ["a"]}).save_to_disk(str(tmp_path / "d"))
    np.savez(tmp_path / "i.npz", embeddings=c.numpy())
    return HipFlatIndex(tmp_path / "d", tmp_path / "i.npz", device="cpu")


def _search(index, by_narrow):
    """Whether the rows in 16 bits were asked; the answer is the corpus's."""
    q = torch.randn(3, 8, generator=torch.Generator().manual_seed(2))
    by_narrow.clear()
    found = index.search(q.numpy(), 4)
    want = (q @ vars(index)["corpus"].t()).topk(4).indices.tolist()
    assert found.total_indices == want
    return len(by_narrow) > 0


@pytest.mark.parametrize("write", [
    lambda c: c.mul_(-1), lambda c: c.data.mul_(-1),
    lambda c: c.numpy().__imul__(-1)], ids=["counted", "data", "memory"])
def test_rows_that_may_have_been_written_to(index, by_narrow, write):
    assert _search(index, by_narrow) and _search(index, by_narrow)
    write(index.corpus)
    assert not _search(index, by_narrow)
    assert index.narrow is None
    index.renew_narrow()
    assert _search(index, by_narrow)


def test_rows_that_were_replaced(index, by_narrow):
    index.corpus = -vars(index)["corpus"]
    assert index.narrow is None and not _search(index, by_narrow)
    index.renew_narrow()
    assert index.narrow.corpus is vars(index)["corpus"]
    assert _search(index, by_narrow)


def test_counted_writes_by_who_has_the_rows(index, by_narrow):
    rows = index.corpus
    index.renew_narrow()
    rows.mul_(-1)
    assert not _search(index, by_narrow) and index.narrow is None


@pytest.mark.parametrize("args", [{"precision": "ubinary"},
                                  {"search_algorithm": "ivf"}])
def test_indices_without(index, tmp_path, by_narrow, args):
    with pytest.warns() if "precision" in args else _nothing():
        other = HipFlatIndex(tmp_path / "d", tmp_path / "i.npz", device="cpu",
                             **args)
    assert other.narrow is None


def test_an_index_told_to_do_without(index, tmp_path, by_narrow):
    paths = tmp_path / "d", tmp_path / "i.npz"
    other = HipFlatIndex(*paths, device="cpu", narrow_rows=False)
    assert other.narrow is None and not _search(other, by_narrow)
    other.renew_narrow()
    assert _search(other, by_narrow)
    config = {"dataset_dir": paths[0], "faiss_index_path": paths[1]}
    for told in ({}, {"narrow_rows": False}):
        args = HipIndexConfig(**config, **told).model_dump(exclude={"name"})
        assert (HipFlatIndex(**args, device="cpu").narrow is None) == bool(told)


def test_no_corpus():
    with pytest.raises(AttributeError):
        HipFlatIndex.__new__(HipFlatIndex).corpus


def test_rows_that_leave_most_questions_are_spared(index, monkeypatch):
    """Searches go without after those that had to ask again for two fifths and
    more, one, two, four, ... of them, until one does better."""
    left, tried = [3], []

    def found(q, corpus, k, narrow, general):
        tried.append(True)
        v, i = general(q, k)
        if left[0] < len(q):
            general(q[: left[0]], k)
        return v.tolist(), i.tolist()

    monkeypatch.setattr(ops, "found_narrow", found)

    def search():
        tried.clear()
        q = torch.randn(5, 8, generator=torch.Generator().manual_seed(2))
        got = index.search(q.numpy(), 4).total_indices
        assert got == (q @ vars(index)["corpus"].t()).topk(4).indices.tolist()
        return bool(tried)

    for pause in (1, 2, 4, 8, 16, 32, 64, 64):
        assert search() and not any(search() for _ in range(pause))
    left[0] = 2
    assert all(search() for _ in range(3))
    left[0] = 3
    assert search() and not search() and search()
    index.renew_narrow()
    assert search()


@pytest.mark.parametrize("Q, N, K, k, by", [
    # own time over the general way's, measured
    (1, 250000, 768, 5, True), (256, 250000, 768, 10, True),  # 0.58, 0.49
    (4, 64, 384, 10, True), (1000, 4000, 1024, 20, True),  # 0.5, 0.94
    (1, 32000, 2048, 60, False), (1, 64000, 2048, 60, True),  # 0.94, 0.82
    (1, 4000, 2048, 60, False), (64, 4000, 8192, 60, False),  # 1.5, 1.9
    (1, 1000, 4096, 1, False), (1, 4000, 8192, 60, False),  # 1.3, 3.5
    (16, 20000, 4096, 60, False), (1, 250000, 4096, 60, True),  # 1.25, 0.77
    (4, 1000, 1536, 20, True), (17, 2000, 1536, 60, False),  # 0.63, 1.13
    (600, 16000, 4096, 20, True), (600, 4000, 8192, 60, False),  # 0.94, 1.6
    (1, 32000, 16384, 10, False), (1000, 1000, 384, 10, False)])  # 1.9, 1.0
def test_where_rows_in_16_bits_are_the_faster_way(Q, N, K, k, by):
    assert ops._narrow_fills(Q, N, K, k) == by


@pytest.mark.skipif(torch.cuda.is_available(), reason="the failure of a host "
                    "without a GPU")
def test_no_pinned_memory():
    """A search then copies its questions; it does not fail."""
    with pytest.raises(RuntimeError):
        torch.empty(64, pin_memory=True)
    assert ops._hip_ops.pinned(64) is None
