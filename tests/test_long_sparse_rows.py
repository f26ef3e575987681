"""Sums over sparse rows in launches of more wavefronts than run at once: the long rows go to workgroups of their own in front
of the others, whole slices of them and single ones, first and last rows, rows at the bound."""
import numpy as np
import pytest

import parpy_amd as parpy
from parpy_amd.compile import hiprtc_compile

HIP = parpy.CompileBackend.Hip


@parpy.jit
def spmv(A, x, y):
    parpy.label('row')
    for row in range(A["nrows"]):
        y[row] = 0.0
        parpy.label('i')
        for i in range(A["rows"][row], A["rows"][row + 1]):
            y[row] += A["values"][i] * x[A["cols"][i]]


def opts(n, tpb=None):
    par = parpy.threads(n)
    o = parpy.par({'row': par.tpb(tpb) if tpb else par})
    o.backend = HIP
    return o


def matrix(n, lengths, dtype, seed=5):
    rng = np.random.default_rng(seed)
    rows = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    nnz = int(rows[-1])
    return {"values": rng.standard_normal(nnz).astype(dtype), "rows": rows, "cols": rng.integers(0, n, nnz), "nrows": n}


def lengths_of(kind, n):
    rng = np.random.default_rng(n)
    lengths = rng.integers(0, 13, n)
    if kind == "ends":
        lengths[[0, 1, n - 1]] = [5000, 257, 4097]
    elif kind == "bound":
        lengths[100:112] = [255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 2047, 2048, 2049]
    elif kind == "slice":
        lengths[3000:3080] = 300          # neighbours: one workgroup in front has them all
    return lengths


def test_long_rows_stand_in_front():
    n = 140001
    A = matrix(n, lengths_of("ends", n), np.float32)
    s = parpy.print_compiled(spmv, [A, np.zeros(n, np.float32), np.zeros(n, np.float32)], opts(n))
    hiprtc_compile(s[:s.index("// host side")], opts(n))
    assert "if (blockIdx.x >= 512) return;" in s and "dim3(512, 1, 1)" in s
    # all at once: as many in front as have room beside the others, none where there is none
    for n, each, in_front in ((20000, 7, 433), (4000, 7, 250), (8000, 150, 0), (65536, 16, 0)):
        A = matrix(n, np.full(n, each), np.float32)
        s = parpy.print_compiled(spmv, [A, np.zeros(n, np.float32), np.zeros(n, np.float32)], opts(n))
        assert (f"if (blockIdx.x >= {in_front}) return;" in s) if in_front else ") return;" not in s, n


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tol", [(np.float32, 2e-5), (np.float64, 1e-13)], ids=["f32", "f64"])
@pytest.mark.parametrize("kind", ["ends", "bound", "slice", "even"])
def test_sums(kind, dtype, tol):
    for n, tpb in ((140001, None), (140001, 128), (131073, 64)):
        A = matrix(n, lengths_of(kind, n), dtype)
        x = np.random.default_rng(1).standard_normal(n).astype(dtype)
        y = np.full(n, -1.0, dtype)
        spmv(A, x, y, opts=opts(n, tpb))
        terms = A["values"].astype(np.float64) * x[A["cols"]]
        want = np.add.reduceat(np.append(terms, 0.0), A["rows"][:-1])
        want[A["rows"][1:] == A["rows"][:-1]] = 0.0
        # rounding of sums of up to 5000 products of size one
        assert np.abs(y - want).max() < tol * np.sqrt(5000) * 4, (n, tpb)


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


def column_opts(n, cols):
    o = parpy.par({'i': parpy.threads(n), 'j': parpy.threads(cols)})
    o.backend = HIP
    return o


def test_elements_of_long_rows_stand_in_lds():
    for n, cols, staged, in_front in ((1000, 256, 2, 125), (1000, 37, 2, 125), (8192, 128, 2, 0), (8100, 128, 2, 512), (20000, 64, 2, 1024), (1000, 4, 0, 125)):
        A = matrix(n, np.full(n, 20), np.float32)
        args = [A, {"values": np.zeros((n, cols), np.float32), "ncols": cols}, np.zeros((n, cols), np.float32)]
        s = parpy.print_compiled(spmm, args, column_opts(n, cols))
        hiprtc_compile(s[:s.index("// host side")], column_opts(n, cols))
        assert s.count(" staged_") - s.count(" staged_next") >= staged and ("staged_" in s) == (staged > 0), (n, cols)
        assert (f"if (blockIdx.x >= {in_front}) return;" in s) if in_front else ") return;" not in s, (n, cols)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["ends", "bound", "slice", "even"])
@pytest.mark.parametrize("n,cols", [(4000, 256), (4000, 37), (8100, 100), (8192, 128), (20000, 64), (4000, 4)])
def test_sums_of_columns(kind, n, cols):
    lengths = lengths_of(kind, n)
    lengths[50:53] = [1023, 1024, 1025]          # whole pieces of a row and one more
    A = matrix(n, lengths, np.float32)
    B = np.random.default_rng(2).standard_normal((n, cols)).astype(np.float32)
    C = np.full((n, cols), -1.0, np.float32)
    spmm(A, {"values": B, "ncols": cols}, C, opts=column_opts(n, cols))
    terms = A["values"].astype(np.float64)[:, None] * B[A["cols"]]
    want = np.add.reduceat(np.vstack([terms, np.zeros((1, cols))]), A["rows"][:-1])
    want[A["rows"][1:] == A["rows"][:-1]] = 0.0
    # rounding of sums of up to 5000 products of size one
    assert np.abs(C - want).max() < 2e-5 * np.sqrt(5000) * 4
