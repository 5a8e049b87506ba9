"""17 <= n <= 32: products as sums of bf16 parts, where bf16 MFMAs read subnormal operands as zero:
the operands are scaled so that no part is subnormal, down to the smallest FP32 values.  Squarings
from the fifth on whose scaled operands reach 2^60 (a low part's product could overflow to the
opposite infinity) are left to the FP32 instructions.

Tolerance: FP32 sums of at most 2n = 64 terms over 7 + s products, each squaring doubling the
relative error: 2^s * 32 * 2^-24 of the Frobenius norm, 2^s * 1.9e-6; measured at most a tenth.
"""

import math

import pytest
import torch

import flash_hypercons as fh
import oracle

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _matrices(n, batch, scale, seed):
    gen = torch.Generator().manual_seed(seed)
    return torch.randn(batch, n, n, generator=gen) * (scale / n**0.5), torch.randn(batch, n, n, generator=gen)


def _exact(a, g):
    """exp(a) and L(a^T, g) in FP64; g is scaled to norm 1 for the block exponential, L being linear in it."""
    a, g = a.double(), g.double()
    size = g.flatten(1).norm(dim=1).clamp_min(2.0**-1000)[:, None, None]
    at, zero = a.mT, torch.zeros_like(a)
    block = torch.cat((torch.cat((at, g / size), -1), torch.cat((zero, at), -1)), -2)
    return torch.linalg.matrix_exp(a), torch.linalg.matrix_exp(block)[:, :a.shape[-1], a.shape[-1]:] * size


def _squarings(a, g=None):
    return torch.ops.flash_hypercons._expm_params(a, g)[0][:, 1].cpu().double()


def _run(a, g):
    x = a.to(DEV).requires_grad_()
    y = fh.matrix_exp(x)
    (dx,) = torch.autograd.grad(y, x, g.to(DEV))
    return (y.detach().cpu(), dx.cpu()), (_squarings(x.detach()), _squarings(x.detach().mT, g.to(DEV)))


def _check(a, g, slack=0.0, factor=1.0):
    for out, s, want in zip(*_run(a, g), _exact(a, g)):
        err = ((out.double() - want).flatten(1).norm(dim=1) - slack) / want.flatten(1).norm(dim=1)
        bound = 2.0**s * 32 * 2.0**-24 * factor
        assert bool((err <= bound).all()), (err / bound).max()


@pytest.mark.parametrize("n", (17, 31, 32))
@pytest.mark.parametrize("scale", (0.05, 1.0, 6.0))
def test_parts_sum_to_fp32(n, scale):
    _check(*_matrices(n, 5, scale, n))


@pytest.mark.parametrize("n", (17, 32))
@pytest.mark.parametrize("power", (-101, -118, -140))
def test_tiny_gradients_and_entries_keep_fp32_precision(n, power):
    a, g = _matrices(n, 4, 1.0, n - power)
    # Subnormal FP32 results round to half a unit of 2^-149 an entry.
    _check(a, g * 2.0**power, slack=n * 2.0**-150)
    # A decoupled pair of tiny entries in an ordinary matrix: exp of the block diag(0.5, 0.25) with
    # an upper right entry t is t (e^0.5 - e^0.25) / 0.25 there.
    t = 2.0 ** max(power, -120)
    a[1] = 0
    a[1, 0, 0], a[1, 1, 1], a[1, 0, 1] = 0.5, 0.25, t
    y = _run(a, g)[0][0][1, 0, 1].item()
    want = t * (torch.tensor(0.5).double().exp() - torch.tensor(0.25).double().exp()).item() / 0.25
    assert abs(y - want) <= 4e-6 * abs(want)


@pytest.mark.parametrize("n", (17, 32))
def test_products_of_small_entries_keep_fp32_precision(n):
    """Entries that only a product of two small ones reaches: exp(a)_02 = a_01 a_12 / 2 for a alone,
    and e^t times that where the diagonal is t.  A few roundings of 2^-24, each doubled by a squaring."""
    for low, high in ((30, 35), (50, 55), (55, 60), (58, 61), (60, 65), (63, 62), (20, 103)):
        a = torch.zeros(2, n, n)
        a[:, 0, 1], a[:, 1, 2] = 1.3 * 2.0**-low, 1.7 * 2.0**-high
        a[1, (0, 1, 2), (0, 1, 2)] = 5.0
        y, s = fh.matrix_exp(a.to(DEV)).cpu(), _squarings(a.to(DEV))
        want = a[:, 0, 1].double() * a[:, 1, 2].double() / 2 * torch.tensor([0.0, 5.0]).double().exp()
        err = (y[:, 0, 2].double() - want).abs() / want
        assert bool((err <= 2.0**s * 32 * 2.0**-24).all()), (low, high, err)


@pytest.mark.parametrize("n", (17, 32))
@pytest.mark.parametrize("shift", (70, 78, 82, 85))
def test_small_results_and_gradients_at_strong_decay(n, shift):
    """exp(-shift I + noise): squarings down to entries of 2^-120, and gradients of 2^-90 to 2^-105
    at -18 I.  The polynomial's value e^-t, t = shift / 2^s <= 3.01, comes from sums of terms up to
    e^t, so its relative error is up to e^2t times larger; an eighth of that is allowed and a sixth
    of the bound measured."""
    a, g = _matrices(n, 4, 0.02, shift + n)
    _check(a - shift * torch.eye(n), g, factor=math.exp(2 * shift / 2**5) / 8)
    _check(a - 18.0 * torch.eye(n), g * 2.0 ** (-shift - 20), slack=n * 2.0**-150, factor=math.exp(2 * 18 / 2**3) / 8)


@pytest.mark.parametrize("n", (18, 32))
def test_many_squarings_in_and_out_of_range(n):
    gen = torch.Generator().manual_seed(n)
    skew = torch.randn(4, n, n, generator=gen)
    skew = (skew - skew.mT) * 8  # s = 7 or more, orthogonal results: the parts all the way
    _check(skew, torch.randn(4, n, n, generator=gen))
    big = torch.zeros(3, n, n)
    for i, top in enumerate((80.0, 88.0, 200.0)):  # 200: finite operands beyond 2^60, then overflow
        big[i].diagonal().copy_(torch.linspace(-1.0, 1.0, n) * top)
    y, s = fh.matrix_exp(big.to(DEV)).cpu(), _squarings(big.to(DEV))
    diag, want = y.diagonal(dim1=-2, dim2=-1).double(), big.double().diagonal(dim1=-2, dim2=-1).exp()
    fits = want < 3.0e38
    # Decaying entries have the factor of the test above, results below 2^-126 a unit of 2^-149.
    decay = torch.exp(-2 * big.double().diagonal(dim1=-2, dim2=-1) / 2.0 ** s[:, None]) / 8
    bound = (2.0**s * 32 * 2.0**-24)[:, None] * decay.clamp_min(1)
    assert bool((((diag - want).abs() <= bound * want + 2.0**-149) | ~fits).all())
    assert diag[2, -1].item() == float("inf")


def _structured(n, batch, scale, seed):
    """Matrices whose products are single terms or short sums."""
    gen = torch.Generator().manual_seed(seed)
    dense, g = torch.randn(batch, n, n, generator=gen) * scale, torch.randn(batch, n, n, generator=gen)
    blocks = torch.block_diag(*[torch.ones(2, 2)] * n)[:n, :n]
    return g, {"diagonal": dense * torch.eye(n), "pairs": dense * blocks,
               "bidiagonal": dense * (torch.eye(n) + torch.ones(n, n).triu(1).tril(1))}


@pytest.mark.parametrize("n", (17, 32))
@pytest.mark.parametrize("scale", (0.5, 3.0, 10.0))
def test_short_sums_are_as_close_to_fp64_as_fp32_chains(n, scale):
    """The mean error over 512 matrices against that of the oracle's FP32 chains: means of 512 differ
    by about 4% (a matrix's error spreads as widely as its mean), so 1.15 of it leaves out a third more."""
    g, kinds = _structured(n, 512, scale, n)
    for kind, a in kinds.items():
        direction = g * (a != 0)
        got = fh.matrix_exp(a.to(DEV)).cpu(), torch.ops.flash_hypercons._frechet(a.to(DEV), direction.to(DEV)).cpu()
        chain = oracle.torch_matrix_exp(a)[0], oracle.torch_frechet(a, direction)[0]
        for ours, theirs, want in zip(got, chain, _exact(a.mT, direction)):
            want = want.mT if ours is got[0] else want
            mean = [((r.double() - want).flatten(1).norm(dim=1) / want.flatten(1).norm(dim=1)).mean() for r in (ours, theirs)]
            assert mean[0] <= 1.15 * mean[1], (kind, mean)
