"""Time loops of element-wise updates, several steps per launch: every number of elements per lane that the lengths and step
counts below lead to, against the plain loop on the host, bit for bit."""
import re

import numpy as np
import pytest

import parpy_amd as parpy
from parpy_amd.compile import hiprtc_compile

HIP = parpy.CompileBackend.Hip


@parpy.jit
def average(A, B, steps):
    for t in range(steps):
        parpy.label('N')
        B[1:-1] = (A[:-2] + A[1:-1] + A[2:]) / 3.0
        parpy.label('N')
        A[2:-3] = (B[1:-4] + B[2:-3] + B[3:-2]) / -7.0


def opts(n):
    o = parpy.par({'N': parpy.threads(n)})
    o.backend = HIP
    return o


# length, steps, element type -> elements per lane
SHAPES = [(600, 4, np.float32, 1), (3000, 7, np.float64, 1), (300000, 9, np.float64, 2), (9001, 40, np.float64, 3), (4099, 90, np.float32, 3),
          (9001, 60, np.float64, 4), (9002, 60, np.float32, 4), (560001, 40, np.float64, 6), (1200001, 49, np.float64, 8),
          (1000003, 49, np.float64, 10), (4000001, 30, np.float32, 10), (1300001, 60, np.float64, 12), (2500001, 120, np.float32, 12)]


@pytest.mark.parametrize("n,steps,dtype,per_lane", SHAPES)
def test_elements_per_lane(n, steps, dtype, per_lane):
    a = np.zeros(n, dtype)
    s = parpy.print_compiled(average, [a, a, steps], opts(n))
    assert int(re.search(r"A_r_\d+\[(\d+)\];", s)[1]) == per_lane
    assert ("parpy_stretch<" in s[s.index('extern "C"'):]) == (per_lane * a.itemsize > 16)
    hiprtc_compile(s[:s.index("// host side")], opts(n))


@pytest.mark.gpu
@pytest.mark.parametrize("n,steps,dtype,per_lane", SHAPES)
def test_bit_for_bit(n, steps, dtype, per_lane):
    rng = np.random.default_rng(n)
    A, B = rng.standard_normal(n).astype(dtype), rng.standard_normal(n).astype(dtype)
    A[n // 2], B[3] = np.inf, -0.0
    x, y = A.copy(), B.copy()
    average(A, B, steps, opts=opts(n))
    with np.errstate(all="ignore"):
        for _ in range(steps):
            y[1:-1] = (x[:-2] + x[1:-1] + x[2:]) / dtype(3.0)
            x[2:-3] = (y[1:-4] + y[2:-3] + y[3:-2]) / dtype(-7.0)
    assert np.array_equal(A, x, equal_nan=True) and np.array_equal(B, y, equal_nan=True)


@parpy.jit
def counts(A, B, steps):
    for t in range(steps):
        parpy.label('N')
        B[1:-1] = 1
        parpy.label('N')
        A[2:-2] = A[2:-2] * 3 + B[1:-3] - B[4:]
        parpy.label('N')
        B[3:-1] = A[4:]


INTEGERS = [(np.int32, np.int32), (np.int64, np.int64), (np.int32, np.int64), (np.int64, np.int32)]


@pytest.mark.parametrize("a,b", INTEGERS)
def test_integers_compile(a, b):
    for n, steps in ((600, 3), (9001, 20)):
        s = parpy.print_compiled(counts, [np.zeros(n, a), np.zeros(n, b), steps], opts(n))
        assert "parpy_blend<" in s[s.index('extern "C"'):]
        hiprtc_compile(s[:s.index("// host side")], opts(n))


@pytest.mark.gpu
@pytest.mark.parametrize("a,b", INTEGERS)
def test_integers(a, b):
    for n, steps in ((600, 3), (9001, 20)):
        rng = np.random.default_rng(n)
        A, B = rng.integers(-9, 9, n).astype(a), rng.integers(-9, 9, n).astype(b)
        x, y = A.copy(), B.copy()
        counts(A, B, steps, opts=opts(n))
        with np.errstate(all="ignore"):
            for _ in range(steps):
                y[1:-1] = 1
                x[2:-2] = x[2:-2] * a(3) + y[1:-3].astype(a) - y[4:].astype(a)
                y[3:-1] = x[4:]
        assert np.array_equal(A, x) and np.array_equal(B, y), (n, steps)


@parpy.jit
def shifts(A, B, steps):
    for t in range(steps):
        parpy.label('N')
        B[1:-1] = A[2:]
        parpy.label('N')
        A[1:-1] = B[:-2]


@parpy.jit
def ten_terms(A, B, steps):
    for t in range(steps):
        parpy.label('N')
        B[5:-5] = (A[:-10] + A[1:-9] - A[2:-8] + A[3:-7] - A[4:-6] + A[6:-4] - A[7:-3] + A[8:-2] - A[9:-1] + A[10:]) * 0.25
        parpy.label('N')
        A[5:-5] = (B[:-10] - B[1:-9] + B[2:-8] - B[3:-7] + B[4:-6] - B[6:-4] + B[7:-3] - B[8:-2] + B[9:-1] - B[10:]) * 0.5


# updates that cost less and more than an average of three: length, steps, element type -> elements per lane of each
WORK = [(403337, 49, np.float64, 4, 6), (1000003, 49, np.float64, 4, 12), (10007, 49, np.float64, 4, 6), (3000001, 10, np.float32, 4, 10)]


@pytest.mark.parametrize("n,steps,dtype,copies,terms", WORK)
def test_elements_per_lane_by_the_work_of_an_update(n, steps, dtype, copies, terms):
    got = {}
    for fn in (shifts, ten_terms):
        a = np.zeros(n, dtype)
        s = parpy.print_compiled(fn, [a, a.copy(), steps], opts(n))
        got[fn] = int(re.search(r"A_r_\d+\[(\d+)\];", s)[1])
    assert got == {shifts: copies, ten_terms: terms}


@pytest.mark.gpu
@pytest.mark.parametrize("n,steps,dtype", [w[:3] for w in WORK])
def test_copies_and_ten_terms(n, steps, dtype):
    rng = np.random.default_rng(n)
    for fn in (shifts, ten_terms):
        A, B = rng.standard_normal(n).astype(dtype), rng.standard_normal(n).astype(dtype)
        x, y = A.copy(), B.copy()
        fn(A, B, steps, opts=opts(n))
        for _ in range(steps):
            if fn is shifts:
                y[1:-1] = x[2:]
                x[1:-1] = y[:-2]
            else:   # sums in the type of the arrays, from the left
                y[5:-5] = (((((((((x[:-10] + x[1:-9]) - x[2:-8]) + x[3:-7]) - x[4:-6]) + x[6:-4]) - x[7:-3]) + x[8:-2]) - x[9:-1]) + x[10:]) * dtype(0.25)
                x[5:-5] = (((((((((y[:-10] - y[1:-9]) + y[2:-8]) - y[3:-7]) + y[4:-6]) - y[6:-4]) + y[7:-3]) - y[8:-2]) + y[9:-1]) - y[10:]) * dtype(0.5)
        assert np.array_equal(A, x) and np.array_equal(B, y), fn


@parpy.jit
def far(A, B, R, N, steps):
    for t in range(steps):
        parpy.label('N')
        for i in range(R, N - R):
            B[i] = (A[i - R] - A[i] + A[i + R]) * 0.5
        parpy.label('N')
        for i in range(R, N - R):
            A[i] = (B[i - R] + B[i] - B[i + R]) * 0.5


# reach, length, steps, element type -> elements per lane (None: a launch per update)
FAR = [(13, 3001, 3, np.float64, 14), (16, 3001, 10, np.float64, 16), (13, 30001, 40, np.float32, 14), (16, 30001, 40, np.float32, 20),
       (24, 30001, 40, np.float32, 24), (28, 3001, 10, np.float32, 28), (32, 30001, 40, np.float32, 32), (32, 1000003, 20, np.float32, 32),
       (16, 3001, 3, np.float32, None), (32, 3001, 3, np.float32, None), (17, 3001, 10, np.float64, None), (33, 3001, 10, np.float32, None)]


@pytest.mark.parametrize("reach,n,steps,dtype,per_lane", FAR)
def test_updates_of_wide_reach(reach, n, steps, dtype, per_lane):
    a = np.zeros(n, dtype)
    s = parpy.print_compiled(far, [a, a.copy(), reach, n, steps], opts(n))
    m = re.search(r"A_r_\d+\[(\d+)\];", s)
    assert (int(m[1]) if m else None) == per_lane
    hiprtc_compile(s[:s.index("// host side")], opts(n))


@pytest.mark.gpu
@pytest.mark.parametrize("reach,n,steps,dtype", [f[:4] for f in FAR if f[4]])
def test_updates_of_wide_reach_bit_for_bit(reach, n, steps, dtype):
    rng = np.random.default_rng(n + reach)
    A, B = rng.standard_normal(n).astype(dtype), rng.standard_normal(n).astype(dtype)
    x, y = A.copy(), B.copy()
    far(A, B, reach, n, steps, opts=opts(n))
    r = reach
    for _ in range(steps):
        y[r:-r] = (x[:-2 * r] - x[r:-r] + x[2 * r:]) * dtype(0.5)
        x[r:-r] = (y[:-2 * r] + y[r:-r] - y[2 * r:]) * dtype(0.5)
    assert np.array_equal(A, x) and np.array_equal(B, y)
