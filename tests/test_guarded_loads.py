"""Loads that a test of the program guards (padding marked by -1, the steps past the end of a sequence) are not issued
ahead of the test by the passes that move loads: their index need only be in bounds where they are evaluated."""
import re

import numpy as np

import parpy_amd as parpy
from parpy_amd.compile import hiprtc_compile
from parpy_amd.operators import float32

HIP = parpy.CompileBackend.Hip


def kernel(f, args, par, **kw):
    o = parpy.par(par)
    o.backend = HIP
    for k, v in kw.items():
        setattr(o, k, v)
    s = parpy.print_compiled(f, args, o)
    s = s[:s.index("// host side")]
    hiprtc_compile(s, o)
    return s[s.rindex('extern "C"'):]


def padded_groups(idx, x, y, N):
    parpy.label('i')
    for i in range(N):
        k = idx[i]
        s = float32(0.0)
        for c in range(4):
            s = s + (x[4 * k + c] if k >= 0 else float32(0.0))
        y[i] = s


def ragged_groups(idx, x, y, N):
    parpy.label('i')
    for i in range(N):
        k = idx[i]
        s = x[4 * k]
        for c in range(1, 4):
            s = s + (x[4 * k + c] if y[i] > float32(0.5) else float32(0.0))
        y[i] = s


def test_four_loads_under_tests_are_not_packed():
    args = [np.zeros(1000, np.int64), np.zeros(4000, np.float32), np.zeros(1000, np.float32), 1000]
    assert "parpy_vec4<float> pk_" not in kernel(padded_groups, args, {'i': parpy.threads(1000)})
    # one of them is read anyhow: the others lie in the same 16 bytes
    assert "parpy_vec4<float> pk_" in kernel(ragged_groups, args, {'i': parpy.threads(1000)})


def padded_steps(data, lens, tab, a, b, N, S, T):
    parpy.label('i')
    for i in range(N):
        parpy.label('s')
        for s in range(S):
            a[i, s] = 0.0
        for t in range(1, T):
            src = a
            dst = b
            if t & 1:
                src = b
                dst = a
            o = data[i, t]
            parpy.label('s')
            for s in range(S):
                dst[i, s] = src[i, (s + 1) % S] + (tab[o, s] if o >= 0 else float32(0.0))


def steps(data, lens, tab, a, b, N, S, T):
    parpy.label('i')
    for i in range(N):
        parpy.label('s')
        for s in range(S):
            a[i, s] = 0.0
        for t in range(1, T):
            src = a
            dst = b
            if t & 1:
                src = b
                dst = a
            o = data[i, t]
            parpy.label('s')
            for s in range(S):
                dst[i, s] = src[i, (s + 1) % S] + tab[o, s]


STEP_ARGS = [np.zeros((8, 50), np.int8), np.zeros(8, np.int64), np.zeros((101, 256), np.float32), np.zeros((8, 256), np.float32), np.zeros((8, 256), np.float32), 8, 256, 50]


def test_rows_read_under_a_test_are_not_fetched_a_step_ahead():
    par = {'i': parpy.threads(8), 's': parpy.threads(256)}
    k = kernel(padded_steps, STEP_ARGS, par)
    assert "row_tab" not in k and re.search(r"o_\d+\) >= 0\) \? (tab_\d+\[|parpy_at\(tab_)", k)
    assert "row_tab" in kernel(steps, STEP_ARGS, par)
