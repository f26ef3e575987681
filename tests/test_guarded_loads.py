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
