"""Token sets and column shares of the stream-mixing kernels (csrc/hc_mix.hip).

A workgroup takes a set of tokens whose size follows the batch, and 1, 2 or 4 of its wavefronts
share a token's columns, by C alone.  Around every edge of both rules, a token's results are those
of the token by itself, bit for bit, and lie within the bounds of their FP32 sums.
"""

import pytest
import torch

from tests.mixcheck import bound_violations, dE_terms
from tests.test_hc_mix import OPS, same_bits


def _columns(n, dtype):
    """C around the share rule's steps: passes of one wavefront are 2 chunks of 64 vectors of 16
    bytes (n <= 4) or, in the backward at n >= 5, two passes of 2 chunks of 64 vectors of 8 bytes."""
    v = 16 // dtype.itemsize
    width = 64 * v * 2
    return [v, width - v, width, 2 * width - v, 2 * width, 4 * width - v, 4 * width, 4 * width + v]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("n", [2, 3, 4, 5, 8])
def test_column_shares_and_set_sizes(n, dtype):
    torch.manual_seed(n)
    for c in _columns(n, dtype):
        # 2 workgroups a compute unit, each of 1, 2 or 4 tokens side by side: batches around one
        # token, one workgroup, one and two slots everywhere, and a last set partly past the batch.
        for b in (1, 3, 4, 5, 511, 513, 2049) if c <= 2048 else (1, 5, 513):
            h = (torch.randn(b, n, n, device="cuda") * 0.5).to(dtype)
            x = torch.randn(b, n, c, device="cuda").to(dtype)
            g = torch.randn(b, n, c, device="cuda").to(dtype)
            if n <= 4:
                run = lambda s: (*OPS._hc_mix_aux(h[s], x[s], None)[::2], *OPS._hc_mix_aux(h[s], x[s], g[s]))  # noqa: E731
                y, e, dx, dh, de = run(slice(None))
            else:
                e = OPS._matrix_exp(h.float())
                run = lambda s: (OPS._hc_apply(e[s], x[s]), *OPS._hc_apply_backward(e[s], x[s], g[s]))  # noqa: E731
                y, dx, de = run(slice(None))
            for t in {0, b // 2, b - 1}:
                whole = (y, e, dx, dh, de) if n <= 4 else (y, dx, de)
                assert all(same_bits(one, all_[t:t + 1]) for one, all_ in zip(run(slice(t, t + 1)), whole)), (c, b, t)
            at = slice(max(0, b - 8), b)
            e64, x64, g64 = e[at].double().cpu(), x[at].double().cpu(), g[at].double().cpu()
            assert bound_violations(y[at], e64 @ x64, e64.abs() @ x64.abs(), n, dtype) == 0, (c, b)
            assert bound_violations(dx[at], e64.mT @ g64, e64.abs().mT @ g64.abs(), n, dtype) == 0, (c, b)
            assert bound_violations(de[at], g64 @ x64.mT, g64.abs() @ x64.abs().mT, dE_terms(c), torch.float32) == 0, (c, b)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("n", [2, 4, 5, 8])
def test_largest_sets_of_narrow_rows(n, dtype):
    """Rows up to 4 KiB are not shared, and a wavefront's tokens grow as rows shrink, to 16 (n <= 4)
    or 8: whole batches against their pieces, which have smaller sets, bit for bit."""
    torch.manual_seed(n)
    for row, b in ((16, 40001), (256, 36863), (512, 33000), (1024, 20000)):
        c = row // dtype.itemsize
        h = (torch.randn(b, n, n, device="cuda") * 0.5).to(dtype)
        x, g = (torch.randn(b, n, c, device="cuda").to(dtype) for _ in range(2))
        if n <= 4:
            run = lambda s: (*OPS._hc_mix_aux(h[s], x[s], None)[::2], *OPS._hc_mix_aux(h[s], x[s], g[s]))  # noqa: E731
        else:
            e = OPS._matrix_exp(h.float())
            run = lambda s: (OPS._hc_apply(e[s], x[s]), *OPS._hc_apply_backward(e[s], x[s], g[s]))  # noqa: E731
        pieces = [run(slice(i, i + 3001)) for i in range(0, b, 3001)]
        for whole, *parts in zip(run(slice(None)), *pieces):
            assert same_bits(whole, torch.cat(parts)), (row, b)
