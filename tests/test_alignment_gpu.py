"""Operands whose storage does not start at a multiple of 16 bytes, for the
kernels that copy whole pieces to LDS: the same numbers as from aligned ones."""
import pytest
import torch

from distllm_amd import ops
from distllm_amd.ops import _hip_ops

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _off(t):
    """t in storage that starts one element late."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    flat[1:] = t.flatten()
    return flat[1:].view(t.shape)


def _rand(*shape, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*shape, device="cuda", generator=g).to(BF16)


def _same(f, *args):
    want = f(*args)
    for i in range(len(args)):
        got = f(*[_off(a) if i == j else a for j, a in enumerate(args)])
        assert torch.equal(got, want), i


def test_paged_attn(device):
    bt = torch.arange(12, dtype=torch.int32, device="cuda").view(2, 6)
    ctx = torch.tensor([90, 17], dtype=torch.int32, device="cuda")
    _same(lambda q, k, v: ops.paged_attn(q, k, v, bt, ctx), _rand(2, 8, 64),
          _rand(12, 2, 16, 64, seed=1), _rand(12, 2, 16, 64, seed=2))
    eight = [_rand(12, 2, 16, 128, seed=n).to(torch.float8_e4m3fn)
             .view(torch.uint8) for n in (1, 2)]
    q = _rand(2, 8, 128)
    _same(lambda k, v: ops.paged_attn(q, k, v, bt, ctx), *eight)
    _same(lambda k, v: ops.paged_attn(q, k, v, bt, ctx),
          _rand(12, 2, 16, 128, seed=1), _rand(12, 2, 16, 128, seed=2))


def test_latent_attn(device):
    bt = torch.arange(12, dtype=torch.int32, device="cuda").view(2, 6)
    ctx = torch.tensor([90, 17], dtype=torch.int32, device="cuda")
    seq = torch.tensor([0, 1], dtype=torch.int32, device="cuda")
    _same(lambda q, c: ops.latent_attn(q, c, bt, seq, ctx, 64, 0.1),
          _rand(2, 20, 128), _rand(12, 16, 128, seed=1))


def test_caches_are_not_copied(device):
    """Pages that start between 16-byte pieces are read where they are."""
    bt = torch.zeros(1, 4, dtype=torch.int32, device="cuda")
    ctx = torch.tensor([50], dtype=torch.int32, device="cuda")
    seq = torch.zeros(1, dtype=torch.int32, device="cuda")
    pages, latents = (_off(torch.zeros(2000, 1, 16, 128, device="cuda",
                                       dtype=BF16)) for _ in range(2))
    eight = _off(torch.zeros(4000, 1, 16, 128, device="cuda",
                             dtype=torch.uint8))
    q = _rand(1, 8, 128)
    for f in (lambda: ops.paged_attn(q, pages, pages, bt, ctx),
              lambda: ops.paged_attn(q, eight, eight, bt, ctx),
              lambda: ops.latent_attn(q, latents[:, 0], bt, seq, ctx, 64,
                                      0.1)):
        f()
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        f()
        used = torch.cuda.max_memory_allocated() - before
        assert used < 4000 * 2048 / 2  # half of the least of them


def test_attn_window(device):
    cu = torch.tensor([0, 100, 130], dtype=torch.int32, device="cuda")
    maps = ops.varlen_block_map(cu)

    def run(q, kv, kr):
        out = torch.zeros(130, 2, 128, device="cuda", dtype=BF16)
        return ops.attn_window(q, kv, out, cu, cu, maps, 40, 0.1, kr)

    q = _rand(130, 2, 128)
    _same(lambda kv, kr: run(q, kv, kr), _rand(130, 2 * 192, seed=1),
          _rand(130, 64, seed=2))


def test_products(device):
    _same(lambda x, w: _hip_ops.decode_gemm(x, w, None, 0), _rand(3, 256),
          _rand(128, 256, seed=1))
    _same(lambda x, w: _hip_ops.decode_gemm(x, w, None, 0, 1), _rand(40, 256),
          _rand(128, 256, seed=1))
    scale = torch.rand(128, device="cuda")
    w = _rand(128, 256, seed=1).to(torch.float8_e4m3fn).view(torch.uint8)
    _same(lambda x, w: ops.gemv_fp8(x, w, scale), _rand(3, 256), w)
