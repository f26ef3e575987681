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
