"""Residual norms on both sides of where a row gets a wave instead of a
workgroup, at sizes of one and of many loads a thread."""

import pytest
import torch

from distllm_amd import ops
from distllm_amd.ops import torch_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rms", [False, True])
@pytest.mark.parametrize("H", [8, 512, 520, 768, 2056, 3064, 3072, 4096, 8192])
@pytest.mark.parametrize("rows", [8, 9, 2048, 2049])
def test_rows(device, rows, H, rms):
    g = torch.Generator(device=device).manual_seed(rows + H)
    x, r = (torch.randn(rows, H, device=device, generator=g)
            .to(torch.bfloat16) for _ in range(2))
    w, b = (torch.randn(H, device=device, generator=g).to(torch.bfloat16)
            for _ in range(2))
    b = None if rms else b
    got = ops.norm_fwd_sum(x, r, w, b, eps=1e-5, rms=rms)
    want = torch_ref.norm_fwd(x, r, w, b, 1e-5, rms, return_sum=True)
    for a, e in zip(got, want):  # a bf16 step of results of a few units
        torch.testing.assert_close(a.float(), e.float(), atol=1e-2, rtol=8e-3)


@pytest.mark.parametrize("rows, H", [
    (512, 1032), (513, 1032), (1499, 2056), (1500, 2056),  # ahead of the sums
    (65536, 1032), (65537, 1032), (65537, 1024),  # workgroup and wave
    (131076, 512), (131077, 520), (300001, 8)])  # waves of more than a row
@pytest.mark.parametrize("res, bias", [(False, False), (True, True)])
def test_all_at_once(device, rows, H, res, bias):
    g = torch.Generator(device=device).manual_seed(rows + H)
    x, r = (torch.randn(rows, H, device=device, generator=g)
            .to(torch.bfloat16) for _ in range(2))
    w, b = (torch.randn(H, device=device, generator=g).to(torch.bfloat16)
            for _ in range(2))
    for rms in (False, True):
        args = (x, r if res else None, w, b if bias else None, 1e-5, rms)
        # a bf16 step, as above
        torch.testing.assert_close(ops.norm_fwd(*args).float(),
                                   torch_ref.norm_fwd(*args).float(),
                                   atol=1e-2, rtol=8e-3)


@pytest.mark.parametrize("rows, H, sums", [
    (2049, 640, True), (3000, 648, True), (3001, 648, True),  # with a sum
    (3000, 1024, True), (16384, 1032, False), (16385, 1032, False),
    (16385, 1536, False), (2048, 1032, False), (2048, 3072, False),
    (2049, 3072, False), (70001, 128, True), (140001, 264, False)])
def test_workgroup_and_wave(device, rows, H, sums):
    """By what a row has beside it; narrow rows, whose weights are asked for in
    every row of a wave's."""
    g = torch.Generator(device=device).manual_seed(rows + H)
    x, r = (torch.randn(rows, H, device=device, generator=g)
            .to(torch.bfloat16) for _ in range(2))
    w, b = (torch.randn(H, device=device, generator=g).to(torch.bfloat16)
            for _ in range(2))
    for rms, bias in ((False, None), (False, b), (True, None), (True, b)):
        if sums:
            got = ops.norm_fwd_sum(x, r, w, bias, eps=1e-5, rms=rms)
        else:
            got = (ops.norm_fwd(x, None, w, bias, 1e-5, rms),)
        want = torch_ref.norm_fwd(x, r if sums else None, w, bias, 1e-5, rms,
                                  return_sum=sums)
        for a, e in zip(got, want if sums else (want,)):  # as above
            torch.testing.assert_close(a.float(), e.float(), atol=1e-2,
                                       rtol=8e-3)
