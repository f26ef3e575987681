"""Loads that a test of the program guards (padding marked by -1, the steps past the end of a sequence) are not issued
ahead of the test by the passes that move loads: their index need only be in bounds where they are evaluated."""
import re

import numpy as np
import pytest

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


def ended_steps(data, lens, tab, a, b, N, S, T):
    parpy.label('i')
    for i in range(N):
        parpy.label('s')
        for s in range(S):
            a[i, s] = 0.0
            b[i, s] = 0.0
        for t in range(1, T):
            src = a
            dst = b
            if t & 1:
                src = b
                dst = a
            o = data[i, t]
            parpy.label('s')
            for s in range(S):
                if t < lens[i]:
                    dst[i, s] = src[i, (s + 1) % S] + tab[o, s]


def offset_steps(data, lens, tab, a, b, N, S, T):
    parpy.label('i')
    for i in range(N):
        parpy.label('s')
        for s in range(S):
            a[i, s] = 0.0
            b[i, s] = 0.0
        for t in range(1, T):
            src = a
            dst = b
            if t & 1:
                src = b
                dst = a
            o = data[i, t]
            parpy.label('s')
            for s in range(S):
                if t < lens[i]:
                    dst[i, s] = src[i, (s + 1) % S] + tab[o - 1, s]


STEP_ARGS = [np.zeros((8, 50), np.int8), np.zeros(8, np.int64), np.zeros((101, 256), np.float32), np.zeros((8, 256), np.float32), np.zeros((8, 256), np.float32), 8, 256, 50]


def test_rows_read_under_a_test_are_not_fetched_a_step_ahead():
    par = {'i': parpy.threads(8), 's': parpy.threads(256)}
    k = kernel(padded_steps, STEP_ARGS, par)
    assert "row_tab" not in k and re.search(r"o_\d+\) >= 0\) \? (tab_\d+\[|parpy_at\(tab_)", k)
    assert "row_tab" in kernel(steps, STEP_ARGS, par)


def test_the_step_past_the_end_selects_nothing():
    """A loop that a read's length ends: the observation and the row fetched in its last step are its own again, and the
    row of the first step is fetched only where there is one."""
    k = kernel(ended_steps, STEP_ARGS, {'i': parpy.threads(8), 's': parpy.threads(256)})
    assert re.search(r"int t_last_\d+ = parpy_max<int64_t>\(parpy_min<int64_t>\(\(t_end_\d+ - \(int64_t\)\(1\)\), ", k)
    assert re.search(r"o_next_\d+ = .*parpy_min<int>\(\(t_\d+ \+ 1\), t_last_\d+\)", k)
    first = k[:k.index("for (int t_")]
    assert re.search(r"o_first_\d+ = \(\(1 < t_end_\d+\) \? o_next_\d+ : \(\(int8_t\)0\)\);", first)
    assert re.search(r"row_tab_\d+\[0\] = tab_\d+\[\(\(\(int\)\(o_first_\d+\) \* 256\)", first) and first.count("row_tab") == 2
    # an index that is more than the observation itself: no number stands for a row that is there
    first = kernel(offset_steps, STEP_ARGS, {'i': parpy.threads(8), 's': parpy.threads(256)})
    first = first[:first.index("for (int t_")]
    assert re.search(r"if \(1 < t_end_\d+\) \{\s*\{[^}]*row_tab_\d+\[0\] = ", first) and first.count("row_tab") == 2


@pytest.mark.gpu
def test_padding_outside_the_table_is_never_used():
    rng = np.random.default_rng(4)
    N, S, T = 40, 256, 50
    data, tab = rng.integers(0, 101, (N, T)).astype(np.int8), rng.standard_normal((101, S)).astype(np.float32)
    lens = rng.integers(2, T + 1, N)
    lens[:5] = 0, 1, 2, T - 1, T
    data[np.arange(T)[None, :] >= lens[:, None]] = -1
    a, b = np.full((N, S), 5.0, np.float32), np.full((N, S), 5.0, np.float32)
    o = parpy.par({'i': parpy.threads(N), 's': parpy.threads(S)})
    o.backend = HIP
    parpy.jit(ended_steps)(data, lens, tab, a, b, N, S, T, opts=o)
    want = [np.zeros((N, S), np.float32), np.zeros((N, S), np.float32)]
    for i in range(N):
        for t in range(1, lens[i]):
            src, dst = (want[1], want[0]) if t & 1 else (want[0], want[1])
            dst[i] = np.roll(src[i], -1) + tab[data[i, t]]
    assert np.array_equal(a, want[0]) and np.array_equal(b, want[1])   # (single additions: the same bits)

    data[rng.random((N, T)) < 0.3] = -1
    par = parpy.par({'i': parpy.threads(N), 's': parpy.threads(S)})
    par.backend = HIP
    b[:] = 0.0
    parpy.jit(padded_steps)(data, lens, tab, a, b, N, S, T, opts=par)
    want = [np.zeros((N, S), np.float32), np.zeros((N, S), np.float32)]
    for t in range(1, T):
        src, dst = (want[1], want[0]) if t & 1 else (want[0], want[1])
        dst[:] = np.roll(src, -1, axis=1) + np.where(data[:, t, None] >= 0, tab[data[:, t]], np.float32(0.0))
    assert np.array_equal(a, want[0]) and np.array_equal(b, want[1])
