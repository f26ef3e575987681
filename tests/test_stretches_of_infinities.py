"""Stretches of time loops whose divisions by constants leave infinite dividends out: what would have been infinite is NaN at
the end and the stretch is computed again, so the results are those of one launch per update, bit for bit."""
import re

import numpy as np
import pytest

import parpy_amd as parpy
from parpy_amd.compile import hiprtc_compile
from parpy_amd.operators import float32, max

HIP = parpy.CompileBackend.Hip


def averages(A, B, K, n, steps):
    for t in range(steps):
        parpy.label('N')
        B[1:-1] = (A[:-2] + A[1:-1] + A[2:]) / 3.0
        parpy.label('N')
        A[1:-1] = (B[:-2] + B[1:-1] + B[2:]) / -49.0


def coefficients(A, B, K, n, steps):
    """A definition in front of the stores, numbers of the iteration, a division by an element beside those by constants."""
    for t in range(steps):
        parpy.label('N')
        for i in range(1, n - 1):
            s = (A[i - 1] - A[i + 1]) / 10.0
            B[i] = s * 2.0 + float32(i % 3) / 7.0 - A[i] / (K[i] + 3.0)
        parpy.label('N')
        for i in range(n - 1):
            A[i] = B[i + 1] / 6.0


def weighted(A, B, K, n, steps):
    """A division by an element, which is 0 / 0 outside the arrays."""
    for t in range(steps):
        parpy.label('N')
        B[1:-1] = (A[:-2] + A[2:]) / 3.0 / K[1:-1]
        parpy.label('N')
        A[1:-1] = (B[:-2] + B[2:]) / 3.0 / K[1:-1]


def largest(A, B, K, n, steps):
    """A maximum drops NaN: nothing at the end would tell."""
    for t in range(steps):
        parpy.label('N')
        for i in range(1, n - 1):
            B[i] = max(A[i - 1] / 3.0, A[i + 1])
        parpy.label('N')
        for i in range(1, n - 1):
            A[i] = B[i] / 3.0


def chosen(A, B, K, n, steps):
    for t in range(steps):
        parpy.label('N')
        for i in range(1, n - 1):
            B[i] = A[i - 1] / 3.0 if A[i] < 1e30 else A[i]
        parpy.label('N')
        for i in range(1, n - 1):
            A[i] = B[i + 1]


def options(n, **kw):
    o = parpy.par({'N': parpy.threads(n)})
    o.backend = HIP
    for k, v in kw.items():
        setattr(o, k, v)
    return o


@pytest.mark.parametrize("fn,left_out", [(averages, True), (coefficients, True), (largest, False), (chosen, False)])
def test_which_updates_leave_infinities_out(fn, left_out):
    n = 5000
    a = [np.zeros(n, np.float32) for _ in range(3)]
    s = parpy.print_compiled(parpy.jit(fn), a + [n, 20], options(n))
    hiprtc_compile(s[:s.index("// host side")], options(n))
    assert "parpy_lane_before(" in s[s.index('extern "C"'):]
    assert (", false>(" in s[s.index('extern "C"'):]) == left_out


def test_nan_outside_the_arrays_does_not_count():
    n = 5003
    s = parpy.print_compiled(parpy.jit(weighted), [np.zeros(n, np.float32) for _ in range(3)] + [n, 20], options(n))
    tests = re.findall(r"(\w)_r_\d+\[e\] != \1_r_\d+\[e\](.*)\);", s)   # in the stretches at the ends
    bounds = re.compile(rf" && at_\d+ \+ e >= 0 && at_\d+ \+ e < {n}")
    assert sorted(t[0] for t in tests) == ["A", "B"] and all(bounds.fullmatch(t[1]) for t in tests)


def test_what_is_no_number_from_the_start():
    n = 200000
    s = parpy.print_compiled(parpy.jit(averages), [np.zeros(n) for _ in range(3)] + [n, 40], options(n))
    # the array that is loaded is looked at, B is not, inside and at the ends
    assert re.findall(r"ballot_w64\(false(?: \|\| parpy_no_number<\d>\((\w)_r_\d+\))*\) == 0", s) == ["A", "A"]
    # then divisions of any dividend, inside without the tests of the ends
    parts = s[s.index('extern "C"'):s.index("// host side")].split("return; }")
    assert len(parts) == 3 and all(", false>(" in p for p in parts[:2]) and ", false>(" not in parts[2]
    inside, ends = re.split(r"\n  \} else \{", parts[2])
    assert "parpy_div_const<" in inside and "parpy_blend" not in inside and "parpy_blend" in ends


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("fn", [averages, coefficients, weighted, largest, chosen])
def test_infinities_and_nan(fn, dtype):
    f = parpy.jit(fn)
    rng = np.random.default_rng(17)
    info = np.finfo(dtype)
    for n, steps in ((700, 9), (5003, 24), (40001, 24)):
        x = (rng.standard_normal((3, n)) * np.exp2(rng.integers(-20, 20, (3, n)))).astype(dtype)
        x[:, rng.integers(0, n, n // 50)] = -0.0
        for special in ([], [np.inf], [-np.inf, np.inf], [np.nan], [info.max, info.max, info.max], [np.inf, np.nan, -info.max, -0.0]):
            y = x.copy()
            for at in (0, n // 2, n - 1, *rng.integers(0, n, 3)):
                for q, v in enumerate(special):
                    y[0, (at + 2 * q) % n] = v
            got, want = y.copy(), y.copy()
            f(*got, n, steps, opts=options(n))
            f(*want, n, steps, opts=options(n, opt_tile_steps=False))
            assert np.array_equal(got, want, equal_nan=True), (n, special)
            number = ~np.isnan(want)
            assert np.array_equal(np.signbit(got[number]), np.signbit(want[number])), (n, special)
