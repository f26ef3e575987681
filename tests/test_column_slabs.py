"""Sums over sparse rows times a matrix whose columns are divided into slabs, a slab to every second, fourth or eighth workgroup:
columns that are no whole number of slabs or vectors, the last workgroups of a slab, rows at the bound of the shared ones."""
import re

import numpy as np
import pytest
import torch

import parpy_amd as parpy
from parpy_amd.compile import hiprtc_compile

HIP = parpy.CompileBackend.Hip


@parpy.jit
def spmm(A, B, C):
    parpy.label('i')
    for i in range(A["nrows"]):
        parpy.label('j')
        for j in range(B["ncols"]):
            C[i, j] = 0.0
            parpy.label('k')
            for k in range(A["rows"][i], A["rows"][i + 1]):
                C[i, j] += A["values"][k] * B["values"][A["cols"][k], j]


@parpy.jit
def spmm_onto(A, B, C, D):
    parpy.label('i')
    for i in range(A["nrows"]):
        parpy.label('j')
        for j in range(B["ncols"]):
            t = C[i, j]
            parpy.label('k')
            for k in range(A["rows"][i], A["rows"][i + 1]):
                t += A["values"][k] * B["values"][A["cols"][k], j]
            C[i, j] = t
            D[i, j] = t * 2.0


@parpy.jit
def spmm_less(A, B, C, D):
    parpy.label('i')
    for i in range(A["nrows"]):
        x = C[i, 0]
        parpy.label('j')
        for j in range(B["ncols"]):
            t = 0.0
            parpy.label('k')
            for k in range(A["rows"][i], A["rows"][i + 1]):
                t += A["values"][k] * B["values"][A["cols"][k], j]
            D[i, j] = t - x


@parpy.jit
def spmm_less_kept(A, B, C):
    parpy.label('i')
    for i in range(A["nrows"]):
        x = C[i, 0]
        parpy.label('j')
        for j in range(B["ncols"]):
            t = 0.0
            parpy.label('k')
            for k in range(A["rows"][i], A["rows"][i + 1]):
                t += A["values"][k] * B["values"][A["cols"][k], j]
            C[i, j] = t - x


@parpy.jit
def spmm_less_flat(A, B, C, D):
    parpy.label('i')
    for i in range(A["nrows"]):
        x = C[i * B["ncols"]]
        parpy.label('j')
        for j in range(B["ncols"]):
            t = 0.0
            parpy.label('k')
            for k in range(A["rows"][i], A["rows"][i + 1]):
                t += A["values"][k] * B["values"][A["cols"][k], j]
            D[i, j] = t - x


@parpy.jit
def spmm_scaled(A, B, w, C):
    parpy.label('i')
    for i in range(A["nrows"]):
        x = w[i]
        parpy.label('j')
        for j in range(B["ncols"]):
            C[i, j] = 0.0
            parpy.label('k')
            for k in range(A["rows"][i], A["rows"][i + 1]):
                C[i, j] += A["values"][k] * B["values"][A["cols"][k], j] * x


def options(n, cols):
    o = parpy.par({'i': parpy.threads(n), 'j': parpy.threads(cols)})
    o.backend = HIP
    return o


def operands(n, avg, cols, dtype, inner=777, seed=3):
    rng = np.random.default_rng(seed)
    lengths = rng.integers(0, 2 * avg + 1, n)
    longest = max(64, 2 * avg)
    lengths[[0, 1, n // 2, n - 2, n - 1]] = [longest, longest + 1, 0, 9 * longest + 5, longest + 1]
    rows = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    nnz = int(rows[-1])
    A = {"values": rng.standard_normal(nnz).astype(dtype), "rows": rows, "cols": rng.integers(0, inner, nnz), "nrows": n}
    return A, {"values": rng.standard_normal((inner, cols)).astype(dtype), "ncols": cols}


def expected(A, B):
    n, v = A["nrows"], A["values"].astype(np.float64)
    want = np.zeros((n, B["ncols"]))
    np.add.at(want, np.repeat(np.arange(n), np.diff(A["rows"])), v[:, None] * B["values"].astype(np.float64)[A["cols"]])
    return want


# the slabs that the rule chooses: average row times columns in units of 3.5 KB, 16 columns at least, lanes not left idle
SHAPES = [(1000, 40, 256, 8), (1001, 20, 256, 4), (700, 64, 100, 4), (900, 30, 200, 4), (515, 70, 101, 4), (2100, 60, 33, 2),
          (8192, 20, 128, 2), (640, 20, 129, 1), (300, 200, 37, 2), (20011, 24, 64, 1), (12000, 9, 256, 2)]


def slabs_in(text):
    m = re.search(r"slab_\d+ = .*% (\d+)\);", text)
    return int(m.group(1)) if m else 1


@pytest.mark.parametrize("n,avg,cols,slabs", SHAPES)
def test_slabs_of_a_shape(n, avg, cols, slabs):
    A = {"values": np.zeros(n * avg, np.float32), "rows": np.arange(n + 1) * avg, "cols": np.zeros(n * avg, np.int64), "nrows": n}
    args = [A, {"values": np.zeros((99, cols), np.float32), "ncols": cols}, np.zeros((n, cols), np.float32)]
    s = parpy.print_compiled(spmm, args, options(n, cols))
    hiprtc_compile(s[:s.index("// host side")], options(n, cols))
    assert slabs_in(s) == slabs


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tol", [(np.float32, 2e-6), (np.float64, 4e-15)], ids=["f32", "f64"])
@pytest.mark.parametrize("n,avg,cols,slabs", SHAPES)
def test_sums_in_slabs(n, avg, cols, slabs, dtype, tol):
    A, B = operands(n, avg, cols, dtype)
    want = expected(A, B)
    C = np.full((n, cols), -7.0, dtype)
    spmm(A, B, C, opts=options(n, cols))
    # rounding of sums of up to 9 * 400 products of size one in some order: 2^-24 (2^-53) times a random walk's length, and twice that
    assert np.abs(C - want).max() < tol * 60 * 8
    C0 = np.random.default_rng(9).standard_normal((n, cols)).astype(dtype)
    C, D = C0.copy(), np.full((n, cols), -7.0, dtype)
    spmm_onto(A, B, C, D, opts=options(n, cols))
    assert np.abs(C - (want + C0)).max() < tol * 60 * 8
    assert np.array_equal(D, C * dtype(2.0))


@pytest.mark.parametrize("n,avg,cols,slabs", SHAPES[:3])
def test_rows_that_read_first_what_they_store(n, avg, cols, slabs):
    A = {"values": np.zeros(n * avg, np.float32), "rows": np.arange(n + 1) * avg, "cols": np.zeros(n * avg, np.int64), "nrows": n}
    B, C = {"values": np.zeros((99, cols), np.float32), "ncols": cols}, np.zeros((n, cols), np.float32)
    listing = lambda fun, *args: parpy.print_compiled(fun, [A, B, *args], options(n, cols))
    for s in (listing(spmm_less_kept, C), listing(spmm_less, C, C.copy()), listing(spmm_less_flat, C.reshape(-1).copy(), C)):
        hiprtc_compile(s[:s.index("// host side")], options(n, cols))
        assert slabs_in(s) == 1
    assert slabs_in(listing(spmm_scaled, np.zeros(n, np.float32), C)) == slabs


@pytest.mark.gpu
@pytest.mark.parametrize("n,avg,cols,slabs", SHAPES[:3])
def test_sums_of_rows_that_read_first(n, avg, cols, slabs):
    A, B = operands(n, avg, cols, np.float32)
    C0 = np.random.default_rng(9).standard_normal((n, cols)).astype(np.float32)
    want = expected(A, B) - C0[:, :1]
    on_gpu = lambda x: torch.from_numpy(x.copy()).cuda()
    A, B = ({k: on_gpu(v) if isinstance(v, np.ndarray) else v for k, v in d.items()} for d in (A, B))
    C = on_gpu(C0)
    spmm_less_kept(A, B, C, opts=options(n, cols))
    assert np.abs(C.cpu().numpy() - want).max() < 2e-6 * 60 * 8   # (as above)
    C = on_gpu(C0)
    spmm_less(A, B, C, C, opts=options(n, cols))
    assert np.abs(C.cpu().numpy() - want).max() < 2e-6 * 60 * 8
    C = on_gpu(C0)
    spmm_less_flat(A, B, C.view(-1), C, opts=options(n, cols))
    assert np.abs(C.cpu().numpy() - want).max() < 2e-6 * 60 * 8
