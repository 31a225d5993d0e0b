"""Inner products by three bf16 parts of each number: edges of the tiles, all
24 bits, numbers that bf16 does not hold."""
import pytest
import torch

from distllm_amd import ops
from distllm_amd.ops import _hip_ops

pytestmark = pytest.mark.gpu


def _unit(n, k, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(n, k, device="cuda", generator=g)
    return x / x.norm(dim=1, keepdim=True)


@pytest.mark.parametrize("Q", [1, 16, 63, 64, 65, 128, 129, 256, 257, 520])
@pytest.mark.parametrize("N, K", [(1, 32), (127, 64), (129, 96), (1000, 384),
                                  (2049, 768)])
def test_against_64_bits(device, Q, N, K):
    """No larger an error than the library's float32 product has (rms, with a
    tenth of room for what differs by chance in a thousand numbers), and no
    number off by more than its float32 sums can be."""
    q, c = _unit(Q, K, Q), _unit(N, K, N)
    out = _hip_ops.score(q, c)
    want = q.double() @ c.double().t()
    own = out.double() - want
    size = q.double().abs() @ c.double().abs().t()
    # 6 K / 32 roundings of a running sum, 2^-24 each, and as many of 2^-24
    # that the products in an instruction lose; left-out parts 3 * 2^-24
    assert (own.abs() <= size * (12 * K / 32 + 3) * 2 ** -24 + 1e-12).all()
    if Q * N > 1000:
        lib = (q @ c.t()).double() - want
        assert own.pow(2).mean() <= 1.21 * lib.pow(2).mean()


def test_all_bits(device):
    """A one in a query picks a number of the corpus, with every bit."""
    c = torch.randn(300, 64, device="cuda") * 1e3
    out = _hip_ops.score(torch.eye(64, device="cuda"), c)
    assert torch.equal(out, c.t())


@pytest.mark.parametrize("K", [256, 288])
def test_all_bits_of_small_numbers(device, K):
    """As test_all_bits, beside numbers of other sizes in the same row."""
    c = torch.randn(300, K, device="cuda") * torch.logspace(
        0, -20, K, device="cuda")
    out = _hip_ops.score(torch.eye(K, device="cuda"), c)
    assert torch.equal(out, c.t())


def test_not_finite(device):
    """Infinities, NaN and numbers that bf16 rounds to infinity come out as
    from float32 sums."""
    q, c = _unit(70, 64, 1), _unit(200, 64, 2)
    c[3, 5], c[64, 0], c[199, 63] = float("inf"), float("nan"), 3.4e38
    q[69, 7] = float("-inf")
    out = _hip_ops.score(q, c)
    want = (q.double() @ c.double().t()).float()
    assert torch.equal(out.isnan(), want.isnan())
    assert torch.equal(out.isinf(), want.isinf())
    torch.testing.assert_close(out, want, equal_nan=True, rtol=1e-5,
                               atol=1e-6)


@pytest.mark.parametrize("Q", [65, 128, 256, 520])
@pytest.mark.parametrize("N, K", [(40000, 256), (40001, 288), (20003, 352)])
def test_many_tiles(device, Q, N, K):
    """Bounds as of test_against_64_bits; infinities and NaN stay where they are."""
    q, c = _unit(Q, K, Q), _unit(N, K, N)
    c[5000:5300, K - 1] = 70.0
    c[N // 3: N // 3 + 100] *= 1e-6
    c[N - 1, 5], c[777, 0] = float("inf"), float("nan")
    out = _hip_ops.score(q, c)
    want = q.double() @ c.double().t()
    size = q.double().abs() @ c.double().abs().t()
    real = want.isfinite()
    bound = size * (12 * K / 32 + 3) * 2 ** -24 + 1e-12
    assert ((out.double() - want).abs() <= bound)[real].all()
    assert torch.equal(out.isnan(), want.isnan())
    assert torch.equal(out.isinf(), want.isinf())


def test_rule(device):
    """Both sides of the rule agree, as do operands that only one takes."""
    for Q, N, K in ((32, 20000, 64), (33, 20000, 64), (40, 16256, 64),
                    (40, 16257, 64), (300, 9000, 96), (300, 9000, 80)):
        q, c = _unit(Q, K, 3), _unit(N, K, 4)
        want = q.double() @ c.double().t()
        for a, b in ((q, c), (q.t().contiguous().t(), c),
                     (q, c.t().contiguous().t())):
            assert (ops.score(a, b).double() - want).abs().max() < 1e-6
    assert ops.score(q[:0], c).shape == (0, 9000)
    assert ops.score(q, c[:0]).shape == (300, 0)
