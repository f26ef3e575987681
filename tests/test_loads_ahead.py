"""Loads of a thread's own iterations that are issued a group of iterations ahead: shortest and longest loops that take it, a
group that is not whole, types, several loads, an index that is picked by a condition; and the loops beside the rule."""
import re

import numpy as np
import pytest

import parpy_amd as parpy
from parpy_amd.compile import hiprtc_compile
from parpy_amd.operators import exp

M = 2048      # threads: two workgroups


@parpy.jit
def one_load(table, a, b, N, M, T):
    parpy.label('r')
    for r in range(2):
        for t in range(1, T):
            src = b
            dst = a
            if t % 2 == 1:
                src = a
                dst = b
            parpy.label('i')
            for i in range(N):
                dst[r, i] = table[(i % M) // 2] + src[r, i]


@parpy.jit
def picked(table, a, b, N, M, T):
    parpy.label('r')
    for r in range(2):
        for t in range(1, T):
            src = b
            dst = a
            if t % 2 == 1:
                src = a
                dst = b
            parpy.label('i')
            for i in range(N):
                at = 0
                at = i + M if i < N - M else i
                dst[r, i] = (table[(i % M) // 2] + src[r, at]) + src[r, i]


@parpy.jit
def three_loads(table, a, b, N, M, T):
    parpy.label('r')
    for r in range(2):
        for t in range(1, T):
            src = b
            dst = a
            if t % 2 == 1:
                src = a
                dst = b
            parpy.label('i')
            for i in range(N):
                dst[r, i] = ((table[(i % M) // 2] + src[r, i]) + src[r, N - 1 - i]) + src[r, (i + M) % N]


@parpy.jit
def in_place(table, a, b, N, M, T):
    parpy.label('r')
    for r in range(2):
        for t in range(1, T):
            src = b
            dst = a
            if t % 2 == 1:
                src = a
                dst = b
            parpy.label('i')
            for i in range(N):
                dst[r, i] = table[(i % M) // 2] + dst[r, i]


@parpy.jit
def from_parameter(table, a, b, N, M):
    parpy.label('i')
    for i in range(N):
        b[0, i] = table[(i % M) // 2] + a[0, i]


@parpy.jit
def with_exponentials(table, a, b, N, M, T):
    parpy.label('r')
    for r in range(2):
        for t in range(1, T):
            src = b
            dst = a
            if t % 2 == 1:
                src = a
                dst = b
            parpy.label('i')
            for i in range(N):
                dst[r, i] = exp(table[(i % M) // 2] + src[r, i])


def opts(threads=M, **kw):
    o = parpy.par({'r': parpy.threads(2), 'i': parpy.threads(threads)})
    o.backend = parpy.CompileBackend.Hip
    o.opt_vectorize = False     # (would take the lengths that are whole vectors)
    for k, v in kw.items():
        setattr(o, k, v)
    return o


def data(per, dtype):
    rng = np.random.default_rng(per)
    mk = (lambda n: rng.integers(-1000, 1000, n).astype(dtype)) if np.dtype(dtype).kind == "i" else (lambda n: rng.standard_normal(n).astype(dtype))
    return mk(M), mk(2 * per * M).reshape(2, per * M), np.zeros((2, per * M), dtype)


def ahead(f, per, dtype=np.float32, n=0, **kw):
    threads = kw.get("threads", M)
    a = np.zeros((2, per * threads), dtype)
    args = [np.zeros(threads, dtype), a, a.copy(), n or per * threads, threads] + ([3] if f is not from_parameter else [])
    s = parpy.print_compiled(f, args, opts(**kw))
    hiprtc_compile(s[:s.index("// host side")], opts(**kw))
    return len(re.findall(r"\w+ ahead_\d+\[\d+\];", s))


def test_which_loops_issue_loads_ahead():
    for per, taken in ((4, 0), (7, 0), (8, 1), (10, 1), (32, 1), (33, 0)):
        assert ahead(one_load, per) == taken, per
    assert ahead(one_load, 9, opt_prefetch_steps=False) == 0
    assert ahead(picked, 9) == 2 and ahead(three_loads, 9) == 3
    assert ahead(in_place, 9) == 0                                                     # stored to by the iterations
    assert ahead(one_load, 9, n=9 * M - 1) == 0                                        # the last iteration is not every thread's
    assert ahead(from_parameter, 9) == 0                                               # the device compiler moves these
    for threads, taken in ((2 ** 18, 1), (2 ** 19, 0)):                                # all at once, two rounds of workgroups
        assert ahead(one_load, 9, threads=threads) == taken and ahead(with_exponentials, 9, threads=threads) == 1
    assert ahead(picked, 9, np.float64) == 2 and ahead(three_loads, 9, np.float64) == 0   # 32 registers, 48


def steps(f, per, table, a, b, T):
    """The same sums, in the order written, on the host."""
    n = per * M
    i = np.arange(n)
    t = np.tile(np.repeat(table[:M // 2], 2), per)
    at = np.where(i < n - M, i + M, i)
    bufs = [b.copy(), a.copy()]
    for step in range(1, T):
        src, dst = bufs[step % 2], bufs[1 - step % 2]
        if f is one_load:
            dst[:] = t + src
        elif f is picked:
            dst[:] = (t + src[:, at]) + src
        elif f is three_loads:
            dst[:] = ((t + src) + src[:, n - 1 - i]) + src[:, (i + M) % n]
        else:
            dst[:] = t + dst
    return bufs[1], bufs[0]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int16], ids=["f32", "f64", "i16"])
@pytest.mark.parametrize("per", [7, 8, 9, 10, 11, 31, 32, 33])
def test_results_are_those_of_the_loads_in_place(per, dtype):
    for f in (one_load, picked, three_loads, in_place):
        for T in (2, 4):
            table, a, b = data(per, dtype)
            want_a, want_b = steps(f, per, table, a, b, T)
            f(table, a, b, per * M, M, T, opts=opts())
            assert np.array_equal(a, want_a) and np.array_equal(b, want_b), (per, f, T)     # the same bits
