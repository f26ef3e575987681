"""Reductions of many short rows, several rows to a workgroup: row counts that leave the last workgroup partly empty, one row too
few and enough of them, one to sixteen wavefronts per row, values that a row adds to; and the kernels beside the rule."""
import re

import numpy as np
import pytest

import parpy_amd as parpy
from parpy_amd.compile import hiprtc_compile
from parpy_amd.operators import exp, max, sum

DTYPES = [np.float32, np.float64]


@parpy.jit
def add_sums(x, out, N):
    parpy.label('i')
    for i in range(N):
        parpy.label('j')
        s = sum(x[i, :])
        out[i] = out[i] + s


@parpy.jit
def largest(x, out, N):
    parpy.label('i')
    for i in range(N):
        parpy.label('j')
        out[i] = max(x[i, :])


@parpy.jit
def chosen(x, pick, out, N):
    parpy.label('i')
    for i in range(N):
        out[i] = -1.0
        if pick[i] > 0:
            parpy.label('j')
            out[i] = sum(x[i, :])


@parpy.jit
def two_loops(x, out, N):
    parpy.label('i')
    for i in range(N):
        parpy.label('j')
        m = max(x[i, :])
        parpy.label('j')
        out[i, :] = exp(x[i, :] - m)


@parpy.jit
def numbers(first, rows, N):
    parpy.label('i')
    for i in range(N):
        parpy.label('j')
        for q in range(first[i], first[i + 1]):
            rows[q] = rows[q] + i


def opts(n, threads):
    o = parpy.par({'i': parpy.threads(n), 'j': parpy.threads(threads)})
    o.backend = parpy.CompileBackend.Hip
    return o


def block(f, args, n, threads):
    s = parpy.print_compiled(f, args, opts(n, threads))
    hiprtc_compile(s[:s.index("// host side")], opts(n, threads))
    return tuple(int(v) for v in re.search(r"<<<dim3\(\d+, \d+, 1\), dim3\((\d+), (\d+), 1\)", s).groups()), s


@pytest.mark.parametrize("n,m,threads,want", [(256, 1000, 64, 1), (257, 700, 64, 8), (5000, 300, 256, 8), (5000, 1500, 256, 8), (5000, 3000, 256, 4),
                                               (5000, 5000, 512, 2), (5000, 30000, 1024, 1), (20000, 3500, 256, 1)])
def test_rows_of_a_workgroup(n, m, threads, want):
    x = np.zeros((n, m), np.float32)
    (width, rows), s = block(add_sums, [x, np.zeros(n, np.float32), n], n, threads)
    assert rows == want and width * rows <= 1024
    assert ("readfirstlane(i_" in s) == (width > 64 and n % rows != 0)      # (a row per wavefront has no barriers)


def test_rows_that_stay_alone():
    for n, m, rows in ((257, 500, 4), (256, 500, 1), (4096, 2000, 1), (4097, 700, 4)):      # a wavefront each, no barriers
        x = np.zeros((n, m), np.float32)
        assert block(two_loops, [x, x.copy(), n], n, 64)[0] == (64, rows), (n, m)
    x, out = np.zeros((5000, 1500), np.float32), np.zeros(5000, np.float32)
    assert block(two_loops, [x, x.copy(), 5000], 5000, 256)[0][1] == 1
    assert block(chosen, [x, np.ones(5000, np.int32), out, 5000], 5000, 256)[0][1] == 1     # a barrier that not every row meets


def test_rows_that_never_meet():
    for n, threads, rows in ((2047, 64, 1), (2048, 64, 8), (5001, 128, 4), (5001, 256, 1)):
        (width, group), s = block(numbers, [np.zeros(n + 1, np.int64), np.zeros(9, np.int64), n], n, threads)
        assert (width, group) == (threads, rows) and ("readfirstlane(i_" in s) == (rows > 1 and n % rows != 0)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2047, 2048, 5001])
def test_row_numbers(n):
    for threads in (64, 128):
        first = np.concatenate([[0], np.cumsum(np.random.default_rng(n).integers(0, 200, n))]).astype(np.int64)
        rows = np.arange(first[-1], dtype=np.int64)
        numbers(first, rows, n, opts=opts(n, threads))
        assert np.array_equal(rows - np.arange(first[-1]), np.repeat(np.arange(n), np.diff(first)))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("n", [257, 1000, 4099])
@pytest.mark.parametrize("m", [200, 777, 2999])
def test_every_row_once(n, m, dtype):
    rng = np.random.default_rng(n + m)
    x, out = rng.standard_normal((n, m)).astype(dtype), rng.standard_normal(n).astype(dtype)
    for threads in (64, 256, 1024):
        got, top = out.copy(), np.zeros(n, dtype)
        add_sums(x, got, n, opts=opts(n, threads))
        largest(x, top, n, opts=opts(n, threads))
        # m terms of order one, partial sums of at most 5 sqrt(m): m * 5 sqrt(m) * eps / 2 at the very most, a tenth of it here
        assert np.abs(got - (out + x.astype(np.float64).sum(1))).max() < 0.25 * m * np.sqrt(m) * np.finfo(dtype).eps
        assert np.array_equal(top, x.max(1))
    pick = rng.integers(0, 2, n).astype(np.int32)
    got = np.zeros(n, dtype)
    chosen(x, pick, got, n, opts=opts(n, 256))
    assert np.array_equal(got == -1.0, pick == 0) and np.allclose(got[pick > 0], x[pick > 0].astype(np.float64).sum(1), atol=0.25 * m * np.sqrt(m) * np.finfo(dtype).eps)


@parpy.jit
def scaled_rows(x, y, N, M):
    parpy.label('i')
    for i in range(N):
        parpy.label('j')
        for j in range(M):
            y[i, j] = x[i, j] * 2.0


@parpy.jit
def row_products(x, w, y, N, M, K):
    parpy.label('i')
    for i in range(N):
        parpy.label('j')
        for j in range(M):
            t = 0.0
            for q in range(K):
                t = t + x[i, q] * w[q, j]
            y[i, j] = t


def test_which_rows_that_never_meet_share():
    for n, m, rows in ((20000, 100, 8), (20000, 128, 8), (8192, 500, 8), (100000, 256, 1), (20000, 500, 1), (2000, 100, 1)):
        x = np.zeros((n, m), np.float32)
        assert block(scaled_rows, [x, x.copy(), n, m], n, 64)[0] == (64, rows), (n, m)
    x, w, y = np.zeros((5000, 256), np.float32), np.zeros((256, 64), np.float32), np.zeros((5000, 64), np.float32)
    s = block(row_products, [x, w, y, 5000, 64, 256], 5000, 64)[1]
    assert "<<<dim3(1, 5000, 1), dim3(64, 1, 1)" in s     # (the row's own values are scalar loads)


@pytest.mark.gpu
def test_element_wise_rows_once():
    for n, m in ((20001, 100), (8193, 500), (2049, 65), (20001, 500)):
        x = np.random.default_rng(m).random((n, m)).astype(np.float32)
        for threads in (64, 128):
            y = np.zeros_like(x)
            scaled_rows(x, y, n, m, opts=opts(n, threads))
            assert np.array_equal(y, x * np.float32(2.0)), (n, m, threads)
