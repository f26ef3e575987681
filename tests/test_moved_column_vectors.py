"""Sums over sparse rows times a matrix whose rows are no whole number of vectors: the last vector of a row of columns is moved to
end with the row, beside others in its slab, in the second vector of a lane; rows at the bound of the shared ones."""
import re

import numpy as np
import pytest
import torch

import parpy_amd as parpy
from parpy_amd.compile import hiprtc_compile
from test_column_slabs import expected, operands, options, slabs_in, spmm, spmm_onto


@parpy.jit
def spmm_twice(A, B, C, D):
    parpy.label('i')
    for i in range(A["nrows"]):
        parpy.label('j')
        for j in range(B["ncols"]):
            t = 0.0
            parpy.label('k')
            for k in range(A["rows"][i], A["rows"][i + 1]):
                t += A["values"][k] * B["values"][A["cols"][k], j]
            C[i, j] = t
            D[i, j] = t * 2.0


@parpy.jit
def apart(A, B, E):
    parpy.label('i')
    for i in range(A["nrows"]):
        parpy.label('j')
        for j in range(B["ncols"]):
            t = 0.0
            parpy.label('k')
            for k in range(A["rows"][i], A["rows"][i + 1]):
                t += A["values"][k] * (B["values"][A["cols"][k], j] - E[i, j])
            E[i, j] = t


@parpy.jit
def apart_into(A, B, E, F):
    parpy.label('i')
    for i in range(A["nrows"]):
        parpy.label('j')
        for j in range(B["ncols"]):
            t = 0.0
            parpy.label('k')
            for k in range(A["rows"][i], A["rows"][i + 1]):
                t += A["values"][k] * (B["values"][A["cols"][k], j] - E[i, j])
            F[i, j] = t


# columns: the fewest, one and three past whole vectors, last slabs of few vectors, two vectors a lane
MOVED = [(900, 20, 17), (900, 12, 33), (2100, 60, 35), (515, 70, 101), (640, 24, 65), (700, 40, 199), (700, 40, 227), (1001, 24, 162),
         (20011, 9, 255), (640, 30, 311), (70, 3, 101)]
# a wavefront to a row of columns and lanes or elements too few, fewer than four vectors, doubles
SINGLE = [(640, 20, 129, np.float32), (20011, 6, 255, np.float32), (8000, 10, 162, np.float32), (900, 20, 15, np.float32), (900, 20, 101, np.float64)]


def moved(text, cols):
    return re.search(r", (?:\(int64_t\)\()?%d\)+ \+ (?:\(int64_t\))?\(c_\d+ %% 4\)" % (cols - 4), text) is not None


def text_of(fun, n, avg, cols, dtype, results):
    A = {"values": np.zeros(n * avg, dtype), "rows": np.arange(n + 1) * avg, "cols": np.zeros(n * avg, np.int64), "nrows": n}
    args = [A, {"values": np.zeros((99, cols), dtype), "ncols": cols}] + [np.zeros((n, cols), dtype) for _ in range(results)]
    s = parpy.print_compiled(fun, args, options(n, cols))
    hiprtc_compile(s[:s.index("// host side")], options(n, cols))
    return s


@pytest.mark.parametrize("n,avg,cols", MOVED)
def test_last_vector_ends_with_the_row(n, avg, cols):
    assert moved(text_of(spmm, n, avg, cols, np.float32, 1), cols)
    assert moved(text_of(spmm_twice, n, avg, cols, np.float32, 2), cols)
    # where a row ends by reading what another lane may have stored, every column has one lane
    assert not moved(text_of(spmm_onto, n, avg, cols, np.float32, 2), cols)


@pytest.mark.parametrize("n,avg,cols,dtype", SINGLE)
def test_columns_that_stay_single(n, avg, cols, dtype):
    assert not moved(text_of(spmm, n, avg, cols, dtype, 1), cols)


# vectors of columns that, cut into as many slabs as the row length asks for, would leave the moved one alone in the last slab
ALONE = [(700, 45, 171), (700, 40, 199), (700, 40, 227)]


@pytest.mark.parametrize("n,avg,cols", ALONE)
def test_shared_columns_are_of_one_slab(n, avg, cols):
    for fun, results in ((spmm, 1), (apart, 1), (apart_into, 2)):
        s = text_of(fun, n, avg, cols, np.float32, results)
        vectors = min([int(v) for v in re.findall(r"slab_\d+ \* (\d+)", s)] or [cols])   # of a slab
        assert moved(s, cols) and slabs_in(s) > 1
        assert (cols - 4) // (4 * vectors) == (cols - 1) // (4 * vectors)


@pytest.mark.gpu
@pytest.mark.parametrize("n,avg,cols", MOVED)
def test_sums_of_moved_vectors(n, avg, cols):
    A, B = operands(n, avg, cols, np.float32)
    want = expected(A, B)
    # rounding of sums of up to 9 * 140 products of size one in some order: 2^-24 times a random walk's length, and twice that
    tol = 2e-6 * 60 * 8
    around = np.full((n + 2, cols), -7.0, np.float32)   # nothing in front of or behind the result is touched
    C = around.copy()
    spmm(A, B, C[1:-1], opts=options(n, cols))
    assert np.abs(C[1:-1] - want).max() < tol
    assert (C[0] == -7.0).all() and (C[-1] == -7.0).all()
    C, D = np.full((n, cols), -7.0, np.float32), np.full((n, cols), -7.0, np.float32)
    spmm_twice(A, B, C, D, opts=options(n, cols))
    assert np.abs(C - want).max() < tol
    assert np.array_equal(D, C * np.float32(2.0))
    C0 = np.random.default_rng(9).standard_normal((n, cols)).astype(np.float32)
    C, D = C0.copy(), np.full((n, cols), -7.0, np.float32)
    spmm_onto(A, B, C, D, opts=options(n, cols))
    assert np.abs(C - (want + C0)).max() < tol
    assert np.array_equal(D, C * np.float32(2.0))


@pytest.mark.gpu
def test_infinities_beside_the_moved_vector():
    n, cols = 640, 65
    A, B = operands(n, 24, cols, np.float32)
    B["values"][5, 60], B["values"][7, 61], B["values"][11, 64] = np.inf, np.nan, -np.inf
    with np.errstate(invalid="ignore"):
        want = expected(A, B)
    C = np.full((n, cols), -7.0, np.float32)
    spmm(A, B, C, opts=options(n, cols))
    assert np.array_equal(np.isnan(C), np.isnan(want)) and np.array_equal(np.isinf(C), np.isinf(want))
    at = np.isfinite(want)
    assert np.abs(C[at] - want[at]).max() < 2e-6 * 60 * 8


@pytest.mark.gpu
@pytest.mark.parametrize("n,avg,cols", ALONE)
def test_sums_that_read_what_the_row_stores(n, avg, cols):
    A, B = operands(n, avg, cols, np.float32)
    E = np.random.default_rng(9).standard_normal((n, cols)).astype(np.float32)
    weight = np.zeros(n)
    np.add.at(weight, np.repeat(np.arange(n), np.diff(A["rows"])), A["values"].astype(np.float64))
    want = expected(A, B) - weight[:, None] * E
    on_gpu = lambda x: torch.from_numpy(x.copy()).cuda()
    A, B = ({k: on_gpu(v) if isinstance(v, np.ndarray) else v for k, v in d.items()} for d in (A, B))
    tol = 2 * 2e-6 * 60 * 8   # as above, of products up to twice the size
    out = on_gpu(E)
    apart(A, B, out, opts=options(n, cols))
    assert np.abs(out.cpu().numpy() - want).max() < tol
    out = on_gpu(E)
    apart_into(A, B, out, out, opts=options(n, cols))
    assert np.abs(out.cpu().numpy() - want).max() < tol
