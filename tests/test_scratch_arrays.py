"""Time loops of element-wise updates whose steps write an array before they read it: stretches inside the arrays neither load it
nor, in launches into the second set of arrays, store it."""
import re

import numpy as np
import pytest

import parpy_amd as parpy
from parpy_amd.compile import hiprtc_compile

HIP = parpy.CompileBackend.Hip


def back_and_forth(A, B, C, n, steps):
    for t in range(steps):
        parpy.label('N')
        B[1:-1] = (A[:-2] + A[1:-1] + A[2:]) / 3.0
        parpy.label('N')
        A[1:-1] = (B[:-2] + B[1:-1] + B[2:]) / 3.0


def two_between(A, B, C, n, steps):
    """Two arrays between; elements at both ends that their updates leave alone."""
    for t in range(steps):
        parpy.label('N')
        for i in range(3, n - 5):
            C[i] = A[i - 1] * 0.5
            B[i] = A[i] - A[i + 1]
        parpy.label('N')
        for i in range(4, n - 6):
            A[i] = (C[i + 1] + B[i - 1]) * 0.75


def own_value(A, B, C, n, steps):
    """B takes part in its own update."""
    for t in range(steps):
        parpy.label('N')
        B[1:-1] = A[:-2] * 0.5 + B[1:-1] * 0.5
        parpy.label('N')
        A[1:-1] = B[1:-1] + B[2:]


def read_first(A, B, C, n, steps):
    """B is read by the step's first update and written by the second."""
    for t in range(steps):
        parpy.label('N')
        A[1:-1] = B[1:-1] * 0.5 + B[2:]
        parpy.label('N')
        B[1:-1] = A[:-2] * 0.5


PROGRAMS = [(back_and_forth, "B"), (two_between, "BC"), (own_value, ""), (read_first, "A")]


def options(n, **kw):
    o = parpy.par({'N': parpy.threads(n)})
    o.backend = HIP
    for k, v in kw.items():
        setattr(o, k, v)
    return o


@pytest.mark.parametrize("fn,scratch", PROGRAMS)
def test_which_arrays(fn, scratch):
    n = 200000
    s = parpy.print_compiled(parpy.jit(fn), [np.zeros(n) for _ in range(3)] + [n, 40], options(n))
    hiprtc_compile(s[:s.index("// host side")], options(n))
    loaded = re.findall(r"::in\((\w)_r_\d+, ", s)
    kept = re.findall(r"if \(keep_\d+\) parpy_stretch<double, \d+>::out\((\w)_r_\d+", s)
    stored = re.findall(r"\n +parpy_stretch<double, \d+>::out\((\w)_r_\d+", s)
    # (a path for finite values and one for any)
    assert sorted(set(kept)) == sorted(scratch) and not set(loaded) & set(scratch) and not set(stored) & set(scratch) and "A" in loaded + kept
    # a launch of no steps hands everything on
    s = parpy.print_compiled(parpy.jit(fn), [np.zeros(n) for _ in range(3)] + [n, 3], options(n))
    assert "keep_" not in s or "0 + " not in s[s.index("// host side"):]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("fn,scratch", PROGRAMS)
def test_values(fn, scratch, dtype):
    f = parpy.jit(fn)
    rng = np.random.default_rng(2)
    for n, steps in ((600, 3), (1500, 9), (9001, 25), (50000, 31), (300001, 12)):
        x = rng.standard_normal((3, n)).astype(dtype)
        for special in (None, np.inf, np.nan):
            y = x.copy()
            if special is not None:
                y[:, [0, n // 3, n - 1]] = special
            got, want = y.copy(), y.copy()
            f(*got, n, steps, opts=options(n))
            f(*want, n, steps, opts=options(n, opt_tile_steps=False))
            # (products and sums may be contracted to fused multiply-adds differently: a rounding per step, of values of size one)
            same = np.isclose(got, want, rtol=4 * steps * np.finfo(dtype).eps, atol=4 * steps * np.finfo(dtype).eps, equal_nan=True)
            assert same.all(), (n, steps, special, np.argwhere(~same)[:4])
