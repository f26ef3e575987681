"""Rows that are no whole number of vectors: the last vector of a counted loop ends with the row, a long loop's vectors begin
where a line of memory does, and neither sees the elements of the next row."""
import re

import numpy as np
import pytest

import parpy_amd as parpy
from parpy_amd import workloads as W
from parpy_amd.compile import hiprtc_compile

torch = pytest.importorskip("torch")


def opts(n, threads):
    return parpy.par({'N': parpy.threads(n), 'M': parpy.threads(threads), 'outer': parpy.threads(n), 'inner': parpy.threads(threads)})


def softmax_text(n, m, threads, dtype=np.float32):
    x = np.zeros((n, m), dtype)
    s = parpy.print_compiled(W.softmax, [x, n, m, x.copy()], opts(n, threads))
    hiprtc_compile(s[:s.index("// host side")], opts(n, threads))
    return s[s.index('extern "C" __global__'):]


def sums_text(n, m, threads, dtype=np.float32):
    s = parpy.print_compiled(W.sum_rows, [np.zeros((n, m), dtype), np.zeros(n, dtype), n], opts(n, threads))
    hiprtc_compile(s[:s.index("// host side")], opts(n, threads))
    return s[s.index('extern "C" __global__'):]


def test_which_rows_take_vectors():
    for m, dtype, taken in ((1001, np.float32, True), (1000, np.float32, False), (777, np.float64, True), (1777, np.float16, True),
                            (202, np.float32, False)):   # (whole vectors; a vector a thread)
        assert ("parpy_vector_within<" in softmax_text(5000, m, 256, dtype)) == taken, (m, dtype)
    assert "_front_" in sums_text(3, 40001, 1024) and "_front_" not in sums_text(3, 40000, 1024)
    assert "_front_" not in sums_text(3, 10001, 1024) and "_front_" not in sums_text(3, 40001, 1024, np.float64)


def test_long_rows_of_several_loops_fit_the_registers():
    assert "dim3(512, 1, 1)" in softmax_text(700, 29553, 256, np.float64) and "dim3(256, 1, 1)" in sums_text(700, 29553, 256, np.float64)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tol", [(torch.float16, 4e-3), (torch.float32, 1e-5), (torch.float64, 1e-12)], ids=["f16", "f32", "f64"])
@pytest.mark.parametrize("n,threads", [(4200, 256), (6, 1024)])
def test_rows_do_not_see_their_neighbours(n, threads, dtype, tol):
    """Every other row holds infinities; the ones between are compared with float64."""
    lengths = (257, 258, 259, 515, 1025, 1026, 1027, 2051, 4097, 4099) + ((40001, 40002, 40003, 40031, 33333) if n < 100 else ())
    for m in lengths:
        g = torch.Generator(device="cuda").manual_seed(m)
        x = torch.randn((n, m), generator=g, device="cuda", dtype=torch.float32).to(dtype)
        x[1::2] = float("inf")
        out = torch.full_like(x, -1.0)
        W.softmax(x, n, m, out, opts=opts(n, threads))
        mine = x[::2].double()
        e = torch.exp(mine - mine.max(1, keepdim=True).values)
        want = e / e.sum(1, keepdim=True)
        assert ((out[::2].double() - want).norm() / want.norm()) < tol, m
        sums = torch.full((n,), -1.0, device="cuda", dtype=dtype)
        W.sum_rows(x, sums, n, opts=opts(n, threads))
        assert torch.allclose(sums[::2].double(), mine.sum(1), rtol=tol, atol=tol * 30), m
        assert torch.isinf(sums[1::2]).all(), m


@parpy.jit
def flat(x, out, rows, N, M):
    parpy.label('N')
    for i in range(N):
        parpy.label('M')
        for j in range(M):
            base = i * M
            at = base + 1
            out[at + j] = x[at + j] + 1.0


@parpy.jit
def every_other(x, out, rows, N, M):
    parpy.label('N')
    for i in range(N):
        parpy.label('M')
        for j in range(M):
            r = i * 2
            out[r, j] = x[r, j] + 1.0


@parpy.jit
def picked(x, out, rows, N, M):
    parpy.label('N')
    for i in range(N):
        parpy.label('M')
        for j in range(M):
            r = rows[i]
            out[i, j] = x[r, j] + 1.0


@parpy.jit
def zigzag(x, out, rows, N, M):
    parpy.label('N')
    for i in range(N):
        parpy.label('M')
        for j in range(M):
            r = (i + j * 3) % N
            out[i, j] = x[r, j] + 1.0


@parpy.jit
def zigzag_assigned(x, out, rows, N, M):
    parpy.label('N')
    for i in range(N):
        r = i
        parpy.label('M')
        for j in range(M):
            r = (i + j * 3) % N
            out[i, j] = x[r, j] + 1.0


def named_rows(name, x, rows, n, m):
    """What the functions above write: the rows of the result, and which rows of it they are."""
    i, j = np.arange(n)[:, None], np.arange(m)[None, :]
    one = x.dtype.type(1.0)
    if name == "flat":
        return x.reshape(-1)[1:1 + n * m].reshape(n, m) + one
    if name == "every_other":
        return x[2 * np.arange(n)] + one
    if name == "picked":
        return x[rows] + one
    return x[(i + j * 3) % n, j] + one


NAMED = [flat, every_other, picked, zigzag, zigzag_assigned]


def named_arrays(fn, n, m, dtype):
    rng = np.random.default_rng(m)
    x = rng.random((2 * n, m)).astype(dtype)
    return x.reshape(-1) if fn is flat else x, rng.permutation(2 * n)[:n].astype(np.int64)


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("threads", [128, 256, 512])
def test_rows_named_inside_the_loop_compile(threads, dtype):
    for fn in NAMED:
        x, rows = named_arrays(fn, 20, 40001, dtype)
        s = parpy.print_compiled(fn, [x, x.copy(), rows, 20, 40001], opts(20, threads))
        hiprtc_compile(s[:s.index("// host side")], opts(20, threads))
        if dtype == np.float32 and threads < 512:   # (the row of a pick is not known, nor is there one row in a zigzag)
            assert ("_front_" in s[s.index('extern "C" __global__'):]) == (fn in (flat, every_other)), fn


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float16, np.float32], ids=["f16", "f32"])
def test_rows_named_inside_the_loop(dtype):
    for fn in NAMED:
        for n, m, threads in ((7, 40001, 128), (20, 20003, 256), (300, 999, 64)):
            x, rows = named_arrays(fn, n, m, dtype)
            out = np.full_like(x, -1.0)
            fn(x, out, rows, n, m, opts=opts(n, threads))
            want = np.full_like(x, -1.0)
            if fn is flat:
                want[1:1 + n * m] = named_rows("flat", x, rows, n, m).reshape(-1)
            else:
                want[2 * np.arange(n) if fn is every_other else np.arange(n)] = named_rows(fn.__name__, x, rows, n, m)
            assert np.array_equal(out, want), (fn.__name__, n, m)


def test_rows_assigned_inside_the_loop_are_loaded_inside_it():
    """A row that every iteration picks anew is not known in front of the vector's elements."""
    x, rows = named_arrays(zigzag_assigned, 20, 1001, np.float32)
    s = parpy.print_compiled(zigzag_assigned, [x, x.copy(), rows, 20, 1001], opts(20, 64))
    hiprtc_compile(s[:s.index("// host side")], opts(20, 64))
    assert "parpy_vector_within<" not in s[s.index('extern "C" __global__'):]


# lengths and threads whose vectors are one to a thread, two, and many (the last trip apart), rows taken by fewer workgroups
FEWER = [(777, 128, 10), (777, 64, 10), (2051, 128, 7), (8195, 128, 30)]


@pytest.mark.parametrize("dtype", [np.float16, np.float32, np.float64])
def test_a_loop_over_rows_says_nothing_about_their_vectors(dtype):
    for m, threads, groups in FEWER:
        x = np.zeros((100, m), dtype)
        o = parpy.par({'N': parpy.threads(groups), 'M': parpy.threads(threads)})
        s = parpy.print_compiled(W.softmax, [x, 100, m, x.copy()], o)
        s = s[s.index('extern "C" __global__'):]
        row = re.search(r"int (i_\d+) = \(\(int\)blockIdx", s)[1]
        assert row + "_k" in s and not re.search(r"\(" + row + r"_k < \d+ \|\|", s) and not re.search(row + r"_k < \d+\)?;\n.*parpy_moved", s)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tol", [(torch.float16, 4e-3), (torch.float32, 1e-5), (torch.float64, 1e-12)], ids=["f16", "f32", "f64"])
def test_rows_taken_by_fewer_workgroups(dtype, tol):
    """As above: every other row holds infinities, and a workgroup takes several rows."""
    n = 100
    for m, threads, groups in FEWER:
        g = torch.Generator(device="cuda").manual_seed(m)
        x = torch.randn((n, m), generator=g, device="cuda", dtype=torch.float32).to(dtype)
        x[1::2] = float("inf")
        out = torch.full_like(x, -1.0)
        W.softmax(x, n, m, out, opts=parpy.par({'N': parpy.threads(groups), 'M': parpy.threads(threads)}))
        mine = x[::2].double()
        e = torch.exp(mine - mine.max(1, keepdim=True).values)
        want = e / e.sum(1, keepdim=True)
        assert ((out[::2].double() - want).norm() / want.norm()) < tol, (m, threads, groups)


@parpy.jit
def steps_of_rows(table, obs, a, b, N, M, T):
    parpy.label('N')
    for i in range(N):
        for t in range(T):
            o = obs[i, t]
            parpy.label('M')
            for j in range(M):
                a[i, j] = table[o, j] - a[i, j] + b[j]


# lengths and threads: one vector to a thread, two, and the last trip apart
STEPS = [(1001, 128), (999, 64), (4099, 256), (515, 64), (2050, 64)]


def steps_arrays(m, dtype, n=6, steps=5):
    rng = np.random.default_rng(m)
    table, a, b = (rng.integers(-20, 20, shape).astype(dtype) for shape in ((7, m), (n, m), (m + 9,)))
    obs = rng.integers(0, 7, (n, steps))
    obs[:, -1] = 6   # (the last row: what is past its end is not the table's)
    return table, obs, a, b


@pytest.mark.parametrize("dtype", [np.float16, np.float32, np.int32])
def test_rows_fetched_in_front_of_a_time_loop_compile(dtype):
    for m, threads in STEPS:
        table, obs, a, b = steps_arrays(m, dtype)
        s = parpy.print_compiled(steps_of_rows, [table, obs, a, b, 6, m, 5], opts(6, threads))
        hiprtc_compile(s[:s.index("// host side")], opts(6, threads))
        s = s[s.index('extern "C" __global__'):]
        assert "row_table_" in s and "inv_b_" in s
        # every vector of the table that may not be whole is tested, in front of the loop and behind each step
        assert len(re.findall(rf"if \(j_\d+ < {m}\) {{\n\s*row_table_", s)) == 2


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float16, np.float32, np.int32], ids=["f16", "f32", "i32"])
def test_rows_fetched_in_front_of_a_time_loop(dtype):
    """Small whole numbers: exact in every type."""
    for m, threads in STEPS:
        table, obs, a, b = steps_arrays(m, dtype)
        want = a.copy()
        for t in range(obs.shape[1]):
            want = table[obs[:, t]] - want + b[:m]
        steps_of_rows(table, obs, a, b, 6, m, 5, opts=opts(6, threads))
        assert np.array_equal(a, want), (m, threads)


@parpy.jit
def one_loop(x, y, N, M):
    parpy.label('N')
    for i in range(N):
        parpy.label('M')
        for j in range(M):
            y[i, j] = x[i, j] + 1.0


@parpy.jit
def two_loops(x, y, N, M):
    parpy.label('N')
    for i in range(N):
        parpy.label('M')
        for j in range(M):
            y[i, j] = x[i, j] + 1.0
        parpy.label('M')
        for j in range(M):
            x[i, j] = y[i, j] - x[i, j] * 2.0


@parpy.jit
def two_loops_apart(x, y, N, M):
    parpy.label('N')
    for i in range(N):
        parpy.label('M')
        for j in range(1, M - 1):
            y[i, j] = x[i, j - 1] - x[i, j + 1]
        parpy.label('M')
        for j in range(2, M - 2):
            x[i, j] = y[i, j - 1] + y[i, j + 1]


@parpy.jit
def ring(x, y, N, M):
    parpy.label('N')
    for i in range(N):
        for t in range(5):
            s = x
            d = y
            if t & 1:
                s = y
                d = x
            parpy.label('M')
            for j in range(M):
                d[i, j] = s[i, (j + 1) % M] - s[i, j // 2]


@parpy.jit
def fourth(x, y, N, M):
    parpy.label('N')
    for i in range(N):
        for t in range(5):
            s = x
            d = y
            if t & 1:
                s = y
                d = x
            parpy.label('M')
            for j in range(M):
                d[i, j] = s[i, (j * 4) % M] - s[i, j]


def walked(fn, x, y, m):
    j = np.arange(m)
    if fn in (one_loop, two_loops):
        y[:] = x + x.dtype.type(1)
        if fn is two_loops:
            x[:] = y - x * x.dtype.type(2)
    elif fn is two_loops_apart:
        y[:, 1:-1] = x[:, :-2] - x[:, 2:]
        x[:, 2:-2] = y[:, 1:-3] + y[:, 3:-1]
    else:
        for t in range(5):
            s, d = (y, x) if t & 1 else (x, y)
            d[:] = s[:, (j + 1) % m] - s[:, j // 2] if fn is ring else s[:, (j * 4) % m] - s


WALKS = [(one_loop, False), (two_loops, True), (two_loops_apart, False), (ring, True), (fourth, False)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_which_loops_take_a_part_of_a_vector(dtype):
    """Rows of which a thread walks its elements twice, or which stand in LDS and are read in order."""
    for m, threads in ((1001, 64), (4099, 256)):
        for fn, taken in WALKS:
            x = np.zeros((5, m), dtype)
            s = parpy.print_compiled(fn, [x, x.copy(), 5, m], opts(5, threads))
            hiprtc_compile(s[:s.index("// host side")], opts(5, threads))
            loops = re.findall(r"\(int j_(q_)?\d+_k = 0", s)
            assert loops and all((q == "q_") == taken for q in loops), (fn, m)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_walks_of_odd_rows(dtype):
    """Small whole numbers: exact in every type."""
    for m, threads in ((129, 64), (257, 64), (1001, 64), (1003, 128), (4099, 256)):
        for fn, _ in WALKS:
            rng = np.random.default_rng(m)
            x, y = (rng.integers(-9, 9, (21, m)).astype(dtype) for _ in range(2))
            want_x, want_y = x.copy(), y.copy()
            walked(fn, want_x, want_y, m)
            fn(x, y, 21, m, opts=opts(21, threads))
            assert np.array_equal(x, want_x) and np.array_equal(y, want_y), (fn, m, threads)
