"""Loops over a row that start or end in different places: what one of them keeps in registers is not the other's element."""
import numpy as np
import pytest

import parpy_amd as parpy
from parpy_amd.compile import hiprtc_compile


@parpy.jit
def two_ranges(x, y, z, N, A, B, C, D):
    parpy.label('N')
    for i in range(N):
        parpy.label('M')
        for j in range(A, B):
            y[i, j] = x[i, j] + x[i, j]
        parpy.label('M')
        for j in range(C, D):
            z[i, j] = x[i, j] - y[i, j]


# element type, threads, the two ranges -> whether the second loop finds its elements in registers
RANGES = [(np.float16, 64, (0, 998), (0, 999), False), (np.float16, 64, (0, 999), (0, 998), False), (np.float16, 64, (0, 999), (0, 999), True),
          (np.float16, 64, (0, 1000), (0, 999), False), (np.float32, 128, (0, 1001), (0, 1002), False), (np.float32, 128, (0, 1003), (0, 1003), True),
          (np.float32, 128, (0, 1000), (1, 1001), False), (np.float32, 128, (1, 1001), (1, 1001), True), (np.float64, 64, (2, 1000), (0, 998), False),
          (np.float64, 128, (1, 1000), (0, 999), False), (np.int32, 64, (0, 61), (0, 64), False), (np.int64, 64, (3, 64), (0, 61), False)]


def options(n, threads):
    return parpy.par({'N': parpy.threads(n), 'M': parpy.threads(threads)})


@pytest.mark.parametrize("dtype,threads,first,second,kept", RANGES)
def test_elements_kept_between_loops(dtype, threads, first, second, kept):
    x = np.zeros((5, 1010), dtype)
    s = parpy.print_compiled(two_ranges, [x, x.copy(), x.copy(), 5, *first, *second], options(5, threads))
    hiprtc_compile(s[:s.index("// host side")], options(5, threads))
    assert ("row_x_" in s) == kept and ("row_y_" in s) == kept


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,threads,first,second", [r[:4] for r in RANGES])
def test_two_ranges(dtype, threads, first, second):
    """Sums and differences of small whole numbers: exact in every type."""
    n = 37
    rng = np.random.default_rng(first[1])
    x, y, z = (rng.integers(-50, 50, (n, 1010)).astype(dtype) for _ in range(3))
    want_y, want_z = y.copy(), z.copy()
    want_y[:, slice(*first)] = 2 * x[:, slice(*first)]
    want_z[:, slice(*second)] = x[:, slice(*second)] - want_y[:, slice(*second)]
    two_ranges(x, y, z, n, *first, *second, opts=options(n, threads))
    assert np.array_equal(y, want_y) and np.array_equal(z, want_z)
