"""Time loops inside a kernel whose steps swap two arrays in memory: elements that all threads read, and those of a trip that a
single thread runs, are those of the step before."""
import numpy as np
import pytest

import parpy_amd as parpy
from parpy_amd.compile import hiprtc_compile


@parpy.jit
def broadcast(a, c, r, N, M, T):
    parpy.label('N')
    for i in range(N):
        for t in range(T):
            s = a
            d = c
            if t & 1:
                s = c
                d = a
            parpy.label('M')
            for j in range(1, M):
                d[i, j] = s[i, (j * 4) % M] - s[i, 5]
            parpy.label('M')
            r[i, t] = parpy.operators.max(d[i, :])


@parpy.jit
def last_thread(a, c, r, N, M, T):
    parpy.label('N')
    for i in range(N):
        for t in range(T):
            s = a
            d = c
            if t & 1:
                s = c
                d = a
            parpy.label('M')
            for j in range(1, M - 1):
                d[i, j] = s[i, (j * 4) % M] - parpy.operators.max(s[i, j], s[i, j - 1])
            parpy.label('M')
            r[i, t] = parpy.operators.max(d[i, :])


@parpy.jit
def whole_rows(a, c, N, M, T):
    parpy.label('N')
    for i in range(N):
        for t in range(T):
            s = a
            d = c
            if t & 1:
                s = c
                d = a
            parpy.label('M')
            for j in range(M):
                d[i, j] = s[i, j] + s[i, 5]


def options(groups, threads):
    return parpy.par({'N': parpy.threads(groups), 'M': parpy.threads(threads)})


# rows, workgroups, length, threads: several rows to a workgroup, or rows that do not fit LDS
SHAPES = [(2, 1, 2051, 512), (3, 1, 2050, 512), (3, 3, 30003, 512), (5, 2, 515, 64)]


def test_pointers_that_change_places_are_no_scalars():
    for fn in (broadcast, last_thread):
        for n, groups, m, threads in SHAPES:
            a = np.zeros((n, m), np.float32)
            s = parpy.print_compiled(fn, [a, a.copy(), np.zeros((n, 7), np.float32), n, m, 7], options(groups, threads))
            hiprtc_compile(s[:s.index("// host side")], options(groups, threads))
            assert s.count("+= parpy_vector_zero();") == 2
    # in LDS there are no scalar loads
    a = np.zeros((5, 515), np.float32)
    s = parpy.print_compiled(whole_rows, [a, a.copy(), 5, 515, 7], options(5, 256))
    assert "lds_a_" in s and "+= parpy_vector_zero();" not in s


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int32, np.int64])
@pytest.mark.parametrize("steps", [4, 7])
def test_elements_of_the_step_before(steps, dtype):
    """Whole numbers below 2^(steps + 3): exact in every type."""
    for n, groups, m, threads in SHAPES:
        for fn in (broadcast, last_thread):
            rng = np.random.default_rng(m)
            a, c = (rng.integers(-4, 5, (n, m)).astype(dtype) for _ in range(2))
            r = np.zeros((n, steps), dtype)
            x, y, z = a.copy(), c.copy(), r.copy()
            fn(a, c, r, n, m, steps, opts=options(groups, threads))
            for t in range(steps):
                s, d = (y, x) if t & 1 else (x, y)
                if fn is broadcast:
                    j = np.arange(1, m)
                    d[:, 1:] = s[:, (j * 4) % m] - s[:, 5:6]
                else:
                    j = np.arange(1, m - 1)
                    d[:, 1:-1] = s[:, (j * 4) % m] - np.maximum(s[:, j], s[:, j - 1])
                z[:, t] = d.max(1)
            assert np.array_equal(a, x) and np.array_equal(c, y) and np.array_equal(r, z), (fn, n, m)
