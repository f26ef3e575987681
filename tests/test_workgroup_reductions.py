"""Reductions over a workgroup: every wavefront's partial result counts, whatever their number, and so does every lane's."""
import numpy as np
import pytest

import parpy_amd as parpy
from parpy_amd.operators import sum, prod, max, min

pytestmark = pytest.mark.gpu


@parpy.jit
def all_four(x, total, product, top, low, N):
    parpy.label('N')
    for i in range(N):
        parpy.label('M')
        total[i] = sum(x[i, :])
        parpy.label('M')
        product[i] = prod(x[i, :])
        parpy.label('M')
        top[i] = max(x[i, :])
        parpy.label('M')
        low[i] = min(x[i, :])


# 1, 2, 3, 4, 5, 8, 10 and 16 wavefronts: one to four steps over their partial results
@pytest.mark.parametrize("threads", [64, 128, 192, 256, 320, 512, 640, 1024])
@pytest.mark.parametrize("dtype", ["float16", "float32", "float64", "int32", "int64"])
def test_every_lane_and_wavefront_counts(threads, dtype):
    import torch
    ty = getattr(torch, dtype)
    n, m = 2 * threads, threads
    # row i holds its largest, its smallest and its only factor other than 1 in column i % m: small whole numbers, exact in all types
    x = torch.ones((n, m), dtype=ty, device="cuda")
    x[torch.arange(m), torch.arange(m)] = 3
    x[torch.arange(m, n), torch.arange(m)] = -2
    outs = [torch.zeros(n, dtype=ty, device="cuda") for _ in range(4)]
    all_four(x, *outs, n, opts=parpy.par({'N': parpy.threads(n), 'M': parpy.threads(threads)}))
    first = torch.arange(n, device="cuda") < m
    for got, (a, b) in zip(outs, ((m + 2, m - 3), (3, -2), (3, 1), (1, -2))):
        assert torch.equal(got, torch.where(first, a, b).to(ty)), (threads, dtype)


@pytest.mark.parametrize("threads", [64, 256, 1024])
@pytest.mark.parametrize("dtype", ["float16", "float32", "float64"])
def test_nan_and_infinities(threads, dtype):
    """A maximum or minimum is of the numbers beside a NaN; rows of infinities keep theirs; sums take all of them."""
    import torch
    ty = getattr(torch, dtype)
    m, inf, nan = threads, float("inf"), float("nan")
    rows = torch.full((6, m), -inf, dtype=ty, device="cuda")
    rows[1] = inf
    rows[2] = nan
    rows[2, m - 1] = 2.0
    rows[3] = -0.0
    rows[4] = -1.0
    rows[4, m // 2] = -inf
    rows[5] = nan
    n = rows.shape[0]
    outs = [torch.zeros(n, dtype=ty, device="cuda") for _ in range(4)]
    all_four(rows, *outs, n, opts=parpy.par({'N': parpy.threads(n), 'M': parpy.threads(threads)}))
    total, product, top, low = (o.cpu().double().numpy() for o in outs)
    np.testing.assert_array_equal(top[:5], [-inf, inf, 2.0, 0.0, -1.0])
    np.testing.assert_array_equal(low[:5], [-inf, inf, 2.0, 0.0, -inf])
    np.testing.assert_array_equal(total, [-inf, inf, nan, 0.0, -inf, nan])
    np.testing.assert_array_equal(product[1:], [inf, nan, 0.0, inf, nan])
