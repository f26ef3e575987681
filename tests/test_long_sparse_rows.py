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
    n = 20000     # all at once: shared where they are
    A = matrix(n, lengths_of("ends", n), np.float32)
    assert ") return;" not in parpy.print_compiled(spmv, [A, np.zeros(n, np.float32), np.zeros(n, np.float32)], opts(n))


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
