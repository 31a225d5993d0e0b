"""Which way calls go, where that can be seen without a GPU: calls that a
special form does not cover reach the general one."""

import pytest
import torch

from distllm_amd import ops
from distllm_amd.models import ModelDims, build_model


@pytest.mark.parametrize("arch", ["esm2", "esmc"])
@pytest.mark.parametrize("packed", ["", "1"])
def test_encoder_without_layers(arch, packed, monkeypatch):
    """Embeddings and the last norm are left."""
    if packed:
        monkeypatch.setenv("DISTLLM_FORCE_VARLEN", packed)
    m = build_model(ModelDims(arch=arch, vocab_size=40, hidden_size=32,
                              num_layers=1, num_heads=2,
                              intermediate_size=64), dtype=torch.float32)
    m.layers = m.layers[:0]
    ids = torch.randint(4, 30, (2, 7))
    mask = torch.ones_like(ids)
    mask[1, 5:] = 0
    out = m(ids, mask)
    assert out.shape == (2, 7, 32)
    # the norm's mean and variance, with its weights as they start
    assert out[0].mean(-1).abs().max() < 1e-5
    assert (out[0].var(-1, unbiased=False) - 1).abs().max() < 0.1


class _OnGpu:
    """What ops.score asks of a float32 matrix on a GPU."""

    is_cuda, dtype = True, torch.float32

    def __init__(self, rows, device="cuda:0", columns=64):
        self.shape, self.device = (rows, columns), torch.device(device)

    def is_contiguous(self):
        return True

    def data_ptr(self):
        return 1 << 20

    def t(self):
        return self

    def __matmul__(self, other):
        if self.device != other.device:
            raise RuntimeError("tensors on two devices")
        return "product"


@pytest.fixture
def kernels(monkeypatch):
    class Ops:
        def require(self, name):
            pass

        def score(self, q, corpus):
            return "kernel"

    monkeypatch.setattr(ops, "_hip_ops", Ops())


def test_score_of_two_devices(kernels):
    """Refused by the product, as ever, and not handed to a kernel."""
    q = _OnGpu(256, "cuda:0")
    assert ops.score(q, _OnGpu(50000, "cuda:0")) == "kernel"
    with pytest.raises(RuntimeError, match="two devices"):
        ops.score(q, _OnGpu(50000, "cuda:1"))


def test_score_of_as_many_rows_as_32_bits_count(kernels):
    """A tile's rows past the last one are counted, too."""
    q = _OnGpu(200, "cuda:0")
    assert ops.score(q, _OnGpu((1 << 31) - 256, "cuda:0")) == "kernel"
    for n in ((1 << 31) - 255, (1 << 31) - 1, 1 << 31):
        assert ops.score(q, _OnGpu(n, "cuda:0")) == "product"


@pytest.mark.parametrize("Q, N, K, way", [
    (256, 250000, 768, "kernel"), (128, 250000, 768, "kernel"),
    (64, 250000, 768, "kernel"), (129, 250000, 768, "product"),
    (257, 250000, 768, "product"), (33, 20000, 1024, "product"),
    (33, 20000, 384, "kernel"), (64, 16384, 4096, "product"),
    (64, 20000, 1024, "product"), (64, 50000, 1024, "kernel"),
    (129, 20000, 128, "kernel"), (257, 20000, 128, "product"),
    (129, 250000, 128, "product"),
    (400, 5000, 64, "product"), (1000, 20000, 768, "kernel"),
    (32, 250000, 768, "product")])
def test_score_where_tiles_fill_the_card(kernels, Q, N, K, way):
    assert ops.score(_OnGpu(Q, columns=K), _OnGpu(N, columns=K)) == way


@pytest.mark.parametrize("Q, N, K, k, way", [
    (256, 250000, 768, 10, "kernels"), (129, 250000, 768, 10, "kernels"),
    (65, 20000, 384, 60, "kernels"), (33, 20000, 768, 1, "kernels"),
    (256, 250000, 768, 61, "scores"), (32, 250000, 768, 10, "scores"),
    (256, 4000, 768, 10, "scores"), (64, 8000, 768, 10, "scores"),
    (400, 8000, 256, 10, "scores"), (400, 10000, 352, 10, "kernels"),
    (513, 7700, 384, 10, "kernels"), (256, 10000, 256, 10, "kernels"),
    (64, 40000, 1536, 10, "scores"), (64, 120000, 1536, 10, "kernels"),
    (256, 250000, 784, 10, "scores"), (300, 50000, 128, 10, "scores")])
def test_topk_of_scores_without_their_matrix(monkeypatch, Q, N, K, k, way):
    class Ops:
        def require(self, name):
            pass

        def score_topk(self, q, corpus, k):
            return "kernels"

    class Scores:
        def contiguous(self):
            return self

    monkeypatch.setattr(ops, "_hip_ops", Ops())
    monkeypatch.setattr(ops, "score", lambda q, corpus: Scores())
    monkeypatch.setattr(ops, "topk", lambda scores, k: "scores")
    assert ops.score_topk(_OnGpu(Q, columns=K), _OnGpu(N, columns=K), k) == way


@pytest.mark.parametrize("Q, N, K, k, way", [
    (1, 250000, 768, 5, "few"), (1, 10000, 64, 30, "few"),
    (2, 10000, 1024, 1, "few"), (2, 20000, 128, 1, "few"),
    (4, 32768, 768, 20, "few"), (3, 10000, 256, 5, "few"),
    (1, 9999, 768, 5, "scores"), (1, 250000, 768, 31, "scores"),
    (1, 250000, 1028, 5, "scores"), (1, 250000, 766, 5, "scores"),
    (2, 250000, 64, 5, "scores"), (4, 32769, 512, 5, "scores"),
    (4, 200000, 768, 5, "few"), (3, 200001, 768, 5, "scores"),
    (3, 20000, 1024, 5, "scores"), (4, 20000, 128, 5, "few"),
    (4, 20000, 124, 5, "scores"), (1, 20000, 60, 5, "scores"),
    (5, 20000, 768, 5, "scores")])
def test_search_of_a_few_queries(monkeypatch, Q, N, K, k, way):
    class Ops:
        def require(self, name):
            pass

        def search_few(self, q, corpus, k):
            return "few"

    class Scores:
        def contiguous(self):
            return self

    monkeypatch.setattr(ops, "_hip_ops", Ops())
    monkeypatch.setattr(ops, "score", lambda q, corpus: Scores())
    monkeypatch.setattr(ops, "topk", lambda scores, k: "scores")
    assert ops.score_topk(_OnGpu(Q, columns=K), _OnGpu(N, columns=K), k) == way


class _Cuda(torch.Tensor):
    is_cuda = True


@pytest.mark.parametrize("choice", ["decode", "blt_fused", "blaslt"])
def test_wide_logits_are_not_measured_in_a_capture(monkeypatch, choice):
    """Capture takes a product whose choice, or whose library algorithm at this
    row count, is not there yet: by the form that needs neither."""
    capturing, took = False, []

    def ran(name):
        def run(x, weight, *rest):
            took.append(name)
            if capturing and name == "blt_fused" and not x.shape[0] in known:
                raise RuntimeError("waits in a capture")
            known.add(x.shape[0])
            return torch.empty(x.shape[0], weight.shape[0],
                               dtype=torch.bfloat16)
        return run

    def synchronize():
        if capturing:
            raise RuntimeError("waits in a capture")

    class Ops:
        def require(self, name):
            pass

        decode_gemm = staticmethod(ran("decode"))

    known = set()
    monkeypatch.setattr(ops, "_hip_ops", Ops())
    monkeypatch.setattr(ops, "_blt_fused_path", ran("blt_fused"))
    monkeypatch.setattr(torch.nn.functional, "linear", ran("blaslt"))
    monkeypatch.setattr(torch.cuda, "synchronize", synchronize)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing",
                        lambda: capturing)
    monkeypatch.setattr(ops, "_GEMM_CHOICE", {})
    monkeypatch.setattr(ops, "_WIDE_RUN", set(), raising=False)
    K, N = 1536, 33024
    w = torch.empty(N, K, dtype=torch.bfloat16).as_subclass(_Cuda)
    x = {M: torch.zeros(M, K, dtype=torch.bfloat16).as_subclass(_Cuda)
         for M in (20, 40)}

    def last(M):
        took.clear()
        assert ops.linear(x[M], w).shape == (M, N)
        return took[-1]

    capturing = True  # nothing ran yet
    assert last(20) == "decode" and not ops._GEMM_CHOICE
    ops._GEMM_CHOICE["dec", 128, N, K, False] = choice
    capturing = False
    assert last(20) == choice
    capturing = True
    assert last(20) == choice
    assert last(40) == "decode"


def test_shares_of_k_are_one_of_the_measured_choices(monkeypatch):
    """Blocks of 64 rows that share K: taken by the choice, and where a graph is
    captured before the size ran, for they need no measurement."""
    capturing, took = False, []

    def ran(name):
        def run(x, weight, *rest):
            took.append(name)
            return torch.empty(x.shape[0], weight.shape[0],
                               dtype=torch.bfloat16)
        return run

    def synchronize():
        assert not capturing

    class Ops:
        mid_gemm_shares = staticmethod(lambda M, N, K: int(M > 64) * 2)
        wide_gemm_tile = staticmethod(lambda *sizes: 0)
        decode_gemm = staticmethod(ran("decode"))
        mid_gemm = staticmethod(ran("mid"))

        def require(self, name):
            pass

    monkeypatch.setattr(ops, "_hip_ops", Ops())
    monkeypatch.setattr(ops, "_own_product", lambda *a: True)
    monkeypatch.setattr(ops, "_blt_fused_path", ran("blt_fused"))
    monkeypatch.setattr(torch.nn.functional, "linear", ran("blaslt"))
    monkeypatch.setattr(torch.cuda, "synchronize", synchronize)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing",
                        lambda: capturing)
    monkeypatch.setattr(ops, "_GEMM_CHOICE", {})
    monkeypatch.setattr(ops, "_WIDE_RUN", set())
    w = torch.empty(4096, 4096, dtype=torch.bfloat16).as_subclass(_Cuda)

    def last(M, act=ops.ACT_NONE):
        took.clear()
        x = torch.zeros(M, 4096, dtype=torch.bfloat16).as_subclass(_Cuda)
        assert ops.linear(x, w, None, act).shape == (M, 4096)
        return took[-1]

    capturing = True
    assert last(80) == "mid" and not ops._GEMM_CHOICE
    capturing = False
    last(80)
    assert {"mid", "decode", "blaslt", "blt_fused"} == set(took)
    (key,) = ops._GEMM_CHOICE
    for choice in ("decode", "blt_fused", "blaslt", "mid"):
        ops._GEMM_CHOICE[key] = choice
        assert last(80) == choice
        capturing = True
        assert last(80) == choice
        assert last(100) == "mid"
        capturing = False
    ops._GEMM_CHOICE[key] = "decode"
    assert last(80, ops.ACT_SILU) == last(300) == "mid"
    monkeypatch.setenv("DISTLLM_GEMM", "decode")
    assert last(200) == "decode"


def test_many_rows_go_by_tiles_and_sums():
    """wide_gemm_tile: sizes that the kernel cannot take, rounds of the card's
    CUs, and what is followed stays with torch."""
    tile = ops._hip_ops.wide_gemm_tile
    for sizes in [(5000, 2200, 768, 0), (5000, 2304, 760, 0),
                  (5000, 2304, 64, 0), (0, 256, 128, 0), (5000, 0, 128, 0),
                  (100000, 1 << 20, 1024, 0), (1 << 29, 1 << 20, 128, 0)]:
        assert tile(*sizes) == 0
    assert tile(12992, 768, 768, 0) == 5   # 246 tiles of 160 rows
    assert tile(8448, 4096, 14336, 0) == 6  # 704 of 192 rows, 2.75 rounds
    assert tile(262144, 2304, 768, 0) == 8
    assert tile(300, 768, 768, 0) == 0     # too few tiles
    assert tile(1000, 3072, 768, 2) == 4   # and enough with an activation
    assert tile(16384, 4096, 4096, 0) == 0  # whole rounds of long sums
    assert tile(16384, 28672, 4096, 4) == 8
    # a round of low tiles reads the weights too often
    assert tile(1500, 4096, 4096, 0) == tile(1025, 6144, 4096, 0) == 0
    assert tile(200, 28672, 4096, 4) == tile(1500, 3840, 1280, 0) == 0
    assert tile(300, 28672, 4096, 4) == 5 and tile(1025, 28672, 4096, 4) == 6
    # K of 1536 and more by the share of the card, shorter ones by tiles
    for act in (1, 2, 3, 4, 5):
        assert tile(700, 4096, 1472, act) == 4  # 96 tiles of 128 rows
        assert tile(700, 4096, 1536, act) == tile(1500, 4096, 1536, act) == 0
        assert tile(1700, 4096, 1536, act) == tile(1700, 4096, 2048, act) == 4
        assert tile(1700, 4096, 2112, act) == 0
        assert tile(2600, 6144, 4096, act) == 4
    # two rounds of tiles of 128 rows
    assert tile(2600, 6144, 1024, 0) == tile(2600, 6144, 4096, 0) == 0
    assert tile(2600, 6144, 960, 0) == 4
    assert tile(3000, 4096, 4096, 0) == 6 and tile(12992, 768, 3072, 0) == 5
    shares = ops._hip_ops.mid_gemm_shares
    for sizes in [(64, 768, 768), (300, 760, 768), (300, 768, 760),
                  (300, 768, 64), (300, 0, 768), (1300, 2304, 768),
                  (300, 4096, 4096), (300, 4096, 14336)]:
        assert shares(*sizes) == 0
    assert shares(300, 2304, 768) == shares(2000, 768, 768) == 1
    assert shares(200, 768, 3072) == 4
    # by both measures the slower ones, and some that are not
    assert shares(600, 3072, 2048) == shares(1000, 2048, 2048) == 0
    assert shares(600, 2048, 2048) == shares(1000, 768, 3072) == 1
    assert shares(200, 1280, 5120) == shares(80, 4096, 4096) == 2
    assert shares(80, 2048, 8192) == 4
    x = torch.zeros(2)
    p = torch.nn.Parameter(x)
    assert ops._recorded(p) and not ops._recorded(x, None)
    with torch.no_grad():
        assert not ops._recorded(x, p)
        assert ops._recorded(type("Sub", (torch.Tensor,), {})(2))
        seen = []
        torch.func.vmap(lambda t: seen.append(ops._recorded(t)) or t)(x)
        with torch.autograd.forward_ad.dual_level():
            seen.append(ops._recorded(x))
        from torch.utils.flop_counter import FlopCounterMode
        with FlopCounterMode(display=False):
            seen.append(ops._recorded(x))
        assert seen == [True] * 3


def test_traces_modes_and_casts_are_followed(monkeypatch):
    """A kernel would be a constant of a trace, unseen by a mode of functions,
    and of bf16 where half precision is asked for."""
    from torch.overrides import TorchFunctionMode

    class Sees(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    x, seen = torch.zeros(2), []

    def f(t):
        seen.append(ops._recorded(t))
        return t + 1

    torch.jit.trace(f, x, check_trace=False)
    with Sees():
        f(x)
    with torch.device("cpu"):
        f(x)
    # (no autocast for a GPU that is not there)
    monkeypatch.setattr(ops, "_autocast", lambda: True)
    for dtype in (torch.float16, torch.bfloat16):
        monkeypatch.setattr(torch, "get_autocast_dtype", lambda kind: dtype)
        f(x)
    assert seen == [True, True, False, True, False]


def test_tokens_outside_the_table_are_refused(monkeypatch):
    """A decode step's rows are torch's to take, where a launch makes their norm as
    elsewhere."""
    class Ops:
        def require(self, name):
            pass

        def step_plan(self, ctx, table, layers, H, HKV, fp8, x, w, eps):
            return torch.zeros(1, 8), torch.zeros(layers, 1), x

    class Cache:
        is_cuda, device, shape = True, torch.device("cpu"), (4, 2, 16, 64)
        dtype = torch.bfloat16

    monkeypatch.setattr(ops, "_hip_ops", Ops())
    emb, w = torch.randn(7, 64).bfloat16(), torch.ones(64).bfloat16()
    ints = torch.ones(2, dtype=torch.int32)
    for dtype in (torch.int32, torch.int64):
        tokens = torch.tensor([-7, 6], dtype=dtype)
        x, h, plan = ops.step_begin(tokens, emb, w, 1e-5, 3, ints, 4, Cache(),
                                    ints[:, None])
        assert torch.equal(x[:, 0], emb[[0, 6]]) and h is x and len(plan) == 3
        for wrong in (7, -8):
            tokens[1] = wrong
            with pytest.raises(IndexError):
                ops.step_begin(tokens, emb, w, 1e-5, 3, ints, 4, Cache(),
                               ints[:, None])
