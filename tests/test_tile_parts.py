"""17 <= n <= 32: products as sums of bf16 parts, and the two places where the kernel leaves them
for the FP32 instructions: entries below 2^-100 (a part would be subnormal, which bf16 MFMAs read
as zero) and squarings from the fifth on whose operands reach 2^60 (a low part's product could
overflow to the opposite infinity).

Tolerance: FP32 sums of at most 2n = 64 terms over 7 + s products, each squaring doubling the
relative error: 2^s * 32 * 2^-24 of the Frobenius norm, 2^s * 1.9e-6; measured at most a tenth.
"""

import pytest
import torch

import flash_hypercons as fh

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


def _run(a, g):
    x = a.to(DEV).requires_grad_()
    y = fh.matrix_exp(x)
    (dx,) = torch.autograd.grad(y, x, g.to(DEV))
    s = (torch.ops.flash_hypercons._expm_params(x.detach())[1].cpu(),
         torch.ops.flash_hypercons._expm_params(x.detach().mT, g.to(DEV))[1].cpu())
    return (y.detach().cpu(), dx.cpu()), s


def _check(a, g, rows=slice(None)):
    for out, s, want in zip(*_run(a, g), _exact(a, g)):
        err = (out.double() - want).flatten(1).norm(dim=1) / want.flatten(1).norm(dim=1)
        bound = 2.0 ** s.double() * 32 * 2.0**-24
        assert bool((err <= bound)[rows].all()), (err / bound)[rows].max()


@pytest.mark.parametrize("n", (17, 31, 32))
@pytest.mark.parametrize("scale", (0.05, 1.0, 6.0))
def test_parts_sum_to_fp32(n, scale):
    _check(*_matrices(n, 5, scale, n))


@pytest.mark.parametrize("n", (17, 32))
@pytest.mark.parametrize("power", (-101, -118, -140))
def test_tiny_gradients_and_entries_keep_fp32_precision(n, power):
    a, g = _matrices(n, 4, 1.0, n - power)
    if power > -126:
        _check(a, g * 2.0**power)
    else:  # subnormal FP32: one unit of 2^-149 an entry and product
        got = _run(a, g * 2.0**power)[0][1].double()
        want = _exact(a, g * 2.0**power)[1]
        assert bool(((got - want).abs() <= 2.0**-149 * 64 * n + want.abs() * 1e-3).all())
    # A decoupled pair of tiny entries in an ordinary matrix: exp of the block diag(0.5, 0.25) with
    # an upper right entry t is t (e^0.5 - e^0.25) / 0.25 there.
    t = 2.0 ** max(power, -120)
    a[1] = 0
    a[1, 0, 0], a[1, 1, 1], a[1, 0, 1] = 0.5, 0.25, t
    y = _run(a, g)[0][0][1, 0, 1].item()
    want = t * (torch.tensor(0.5).double().exp() - torch.tensor(0.25).double().exp()).item() / 0.25
    assert abs(y - want) <= 4e-6 * abs(want)


@pytest.mark.parametrize("n", (18, 32))
def test_many_squarings_in_and_out_of_range(n):
    gen = torch.Generator().manual_seed(n)
    skew = torch.randn(4, n, n, generator=gen)
    skew = (skew - skew.mT) * 8  # s = 7 or more, orthogonal results: the parts all the way
    _check(skew, torch.randn(4, n, n, generator=gen))
    big = torch.zeros(3, n, n)
    for i, top in enumerate((80.0, 88.0, 200.0)):  # 200: finite operands beyond 2^60, then overflow
        big[i].diagonal().copy_(torch.linspace(-1.0, 1.0, n) * top)
    y, s = fh.matrix_exp(big.to(DEV)).cpu(), torch.ops.flash_hypercons._expm_params(big.to(DEV))[1].cpu()
    diag, want = y.diagonal(dim1=-2, dim2=-1).double(), big.double().diagonal(dim1=-2, dim2=-1).exp()
    fits = want < 3.0e38
    normal = fits & (want > 2.0**-100)
    bound = (2.0 ** s.double() * 32 * 2.0**-24)[:, None]
    assert bool((((diag - want).abs() <= bound * want) | ~normal).all())
    assert bool((diag[:2] > -1e-30).all()) and not bool(diag[:2].isnan().any())
    assert diag[2, -1].item() == float("inf")
