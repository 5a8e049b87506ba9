"""Stream mixing (n <= 4) over rows of whole dwords that are no whole number of 16-byte vectors.

The kernels' ragged variants read such rows in place.  Zero columns appended up to a whole number
of vectors change no result bit -- they add +0 terms to dE and columns to y and dx -- so the padded
call is the general path to compare with, bit for bit, over the forms an operand can have: any
C around the edges of vectors and passes, dword-aligned slices, 2-byte-aligned 16-bit slices
(copied), strided tokens, broadcast tokens, lazily negated views, single tokens and columns.
"""

import pytest
import torch

from tests.test_hc_mix import OPS, same_bits

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16, torch.float16]


def _padded(t):
    v = 16 // t.element_size()
    return torch.nn.functional.pad(t.contiguous(), (0, -t.shape[2] % v)).resolve_neg()


def _check(h, x, g, what):
    c = x.shape[2]
    y, _, e = OPS._hc_mix_aux(h, x, None)
    dx, dh, de = OPS._hc_mix_aux(h, x, g)
    xp, gp = _padded(x), _padded(g)
    yp, _, ep = OPS._hc_mix_aux(h, xp, None)
    dxp, dhp, dep = OPS._hc_mix_aux(h, xp, gp)
    assert y.is_contiguous() and dx.is_contiguous() and y.shape == x.shape
    pairs = ((y, yp[..., :c]), (e, ep), (dx, dxp[..., :c]), (dh, dhp), (de, dep))
    assert all(same_bits(a, b.contiguous()) for a, b in pairs), what


def _random(shape, dtype):
    return torch.randn(shape, device="cuda").to(dtype)


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("n", [2, 3, 4])
def test_widths(n, dtype):
    torch.manual_seed(n)
    step = 4 // dtype.itemsize  # whole dwords; other widths stay on the padded path
    v = 16 // dtype.itemsize
    width = 64 * v * 2  # one pass of one wavefront; rows of 2 and 4 passes are shared
    # Rows of one chunk of 64 vectors have a path of their own in the forward.
    for c in (step, 2 * step, v - step, v + step, width // 2 - step, width // 2 + step, width - step, width + step,
              2 * width - step, 2 * width + step, 4 * width - step, 4 * width + step):
        for b in (1, 5, 513) if c < 2 * width else (3,):
            _check(_random((b, n, n), dtype) * 0.5, _random((b, n, c), dtype), _random((b, n, c), dtype), (c, b))


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
def test_views(dtype):
    torch.manual_seed(3)
    b, n, c = 7, 3, 514 if dtype != torch.float32 else 1027
    h, g = _random((b, n, n), dtype) * 0.5, _random((b, n, c), dtype)
    for lead in (1, 2, 3):
        wide = _random((b, n, c + 5 + lead), dtype)
        _check(h, wide[..., lead:lead + c], g, ("slice", lead))
        _check(h, g, wide[..., lead:lead + c], ("gradient slice", lead))
    _check(h, _random((n, b, c), dtype).transpose(0, 1), g, "streams first")
    _check(h, _random((b, c, n), dtype).transpose(1, 2), g, "columns first")
    _check(h, _random((1, n, c), dtype).expand(b, n, c), g, "one token for all")
    flat = _random((n * c + 1,), dtype)
    _check(h[:1], flat[1:].as_strided((1, n, c), (n * c + 1, c, 1), 1), g[:1], "odd stride of a single token")
    if dtype == torch.float32:
        neg = torch.complex(g, _random((b, n, c), dtype)).conj().imag
        assert neg.is_neg()
        _check(h, neg, g, "negated view")
        one = _random((b, n, 3), dtype)[..., 1:2]
        _check(h, one, _random((b, n, 1), dtype), "one column")


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
def test_neighbours_of_the_rows_are_left_alone(dtype):
    """Infinite and NaN entries around a slice reach no result."""
    torch.manual_seed(5)
    b, n, c = 6, 4, 130 if dtype != torch.float32 else 129
    h = _random((b, n, n), dtype) * 0.5
    x, g = (torch.full((b, n, c + 8), fill, device="cuda", dtype=dtype) for fill in (float("inf"), float("nan")))
    x[..., 2:2 + c], g[..., 4:4 + c] = _random((b, n, c), dtype), _random((b, n, c), dtype)
    _check(h, x[..., 2:2 + c], g[..., 4:4 + c], "neighbours")
    assert all(bool(t.isfinite().all()) for t in OPS._hc_mix_aux(h, x[..., 2:2 + c], g[..., 4:4 + c]))
