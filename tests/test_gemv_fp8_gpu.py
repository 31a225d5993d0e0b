"""Products with 8-bit weights at the edges of the ring form: one and many
chunks of K, fewer chunks than waves or buffers, ragged columns, every row
count, gated units; and K that it leaves to the general form."""

import pytest
import torch

from distllm_amd import ops

pytestmark = pytest.mark.gpu


def _inputs(M, N, K, device):
    g = torch.Generator(device=device).manual_seed(M * N + K)
    x = torch.randn(M, K, device=device, generator=g).to(torch.bfloat16)
    w = torch.randn(N, K, device=device, generator=g) * K ** -0.5
    wq, s = ops.quantize_fp8_rows(w)
    z = (x.double() @ wq.view(torch.float8_e4m3fn).double().T
         * s.double()).float()
    return x, wq, s, z


def _close(out, ref):  # fp32 sums, one rounding to bf16
    torch.testing.assert_close(out.float(), ref, atol=4e-3, rtol=8e-3)


@pytest.mark.parametrize("N,K", [(16, 128), (7, 256), (100, 640), (64, 80),
                                 (48, 2048), (130, 1152), (33, 16)])
@pytest.mark.parametrize("M", [1, 2, 5, 8])
def test_forms(device, M, N, K):
    x, wq, s, z = _inputs(M, N, K, device)
    b = torch.randn(N, device=device).to(torch.bfloat16)
    _close(ops.gemv_fp8(x, wq, s), z)
    _close(ops.gemv_fp8(x, wq, s, b), z + b.float())


@pytest.mark.parametrize("I,K", [(16, 128), (24, 384), (200, 1024), (8, 80)])
@pytest.mark.parametrize("M", [1, 3, 8])
def test_gated(device, M, I, K):
    x, wq, s, z = _inputs(M, 2 * I, K, device)
    out = ops.gateup_swiglu_fp8(x, wq, s)
    want = torch.nn.functional.silu(z[:, :I]) * z[:, I:]
    torch.testing.assert_close(out.float(), want, atol=2e-2, rtol=1.6e-2)


@pytest.mark.parametrize("N,K", [(512, 4096), (513, 4096), (512, 3968),
                                 (5, 16384), (3, 4224)])
@pytest.mark.parametrize("M", [1, 2])
def test_few_columns(device, M, N, K):
    """Both sides of where one row goes by column."""
    x, wq, s, z = _inputs(M, N, K, device)
    b = torch.randn(N, device=device).to(torch.bfloat16)
    _close(ops.gemv_fp8(x, wq, s, b), z + b.float())
