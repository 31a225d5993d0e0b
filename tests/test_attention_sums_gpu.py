"""The sum of a row's weights in flash attention: one running sum, to which every tile
of 64 keys adds its own."""

import numpy as np
import pytest
import torch

from distllm_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles", [2, 257])
def test_running_sum(device, tiles):
    """Weights are powers of two: 1 for the first tile's keys 0 to 3 of every eight,
    which one half of the lanes has, 2^-25 for all others. Their values sum to 259,
    over 32 the middle of two bf16 numbers, so that the output shows whether a tile's
    2^-19, half a unit of the sum, was added to the whole of it and rounded away."""
    scale = np.float32(np.log(2))
    while scale * np.float32(1.4426950408889634) != 1:
        scale = np.nextafter(scale, np.float32(1 if scale * np.float32(
            1.4426950408889634) < 1 else 0))
    n = 64 * tiles
    one = (torch.arange(n) < 64) & (torch.arange(n) % 8 < 4)
    q = torch.zeros(1, 1, 1, 64)
    q[..., 0] = 1
    k = torch.zeros(1, n, 1, 64)
    k[0, ~one, 0, 0] = -25
    v = torch.zeros(1, n, 1, 64)
    v[0, one] = 8
    v[0, 0] = 11
    want = np.float32(0)
    for t in range(tiles):
        few = int(one[t * 64: t * 64 + 64].sum())
        want += np.float32(few) + np.float32((64 - few) * 2.0 ** -25)
    want = torch.tensor(np.float32(259) * (np.float32(1) / want)).bfloat16()
    out = ops.attn_fwd(*(t.to(device, torch.bfloat16) for t in (q, k, v)),
                       scale=float(scale))
    assert (out.cpu() == want).all()
