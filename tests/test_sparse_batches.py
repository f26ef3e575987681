"""Sums over many sparse rows: two elements in flight per lane (doubles, average rows of 33 to 64) and eight (long average rows),
rows around the batches of a team, empty ones and those that go to the workgroups in front."""
import re

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


def options(n):
    o = parpy.par({'row': parpy.threads(n)})
    o.backend = HIP
    return o


def matrix(n, avg, dtype):
    rng = np.random.default_rng(n)
    lengths = rng.integers(0, 2 * avg + 1, n)
    edges = [0, 1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 4096, 9001]
    lengths[rng.choice(n, len(edges), replace=False)] = edges
    lengths[[0, n - 1]] = 257, 65
    rows = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    return {"values": rng.standard_normal(rows[-1]).astype(dtype), "rows": rows, "cols": rng.integers(0, n, rows[-1]), "nrows": n}


# rows, average, type, lanes of a row, elements in flight
SHAPES = [(57400, 40, np.float64, 32, 2), (57400, 40, np.float32, 32, 4), (57300, 40, np.float64, 32, 4), (57400, 20, np.float64, 16, 4),
          (32800, 140, np.float32, 32, 8), (32800, 140, np.float64, 64, 4), (32800, 170, np.float64, 32, 8), (32700, 140, np.float32, 64, 4)]


@pytest.mark.parametrize("n,avg,dtype,lanes,flight", SHAPES)
def test_batches(n, avg, dtype, lanes, flight):
    A = {"values": np.zeros(n * avg, dtype), "rows": np.arange(n + 1) * avg, "cols": np.zeros(n * avg, np.int64), "nrows": n}
    s = parpy.print_compiled(spmv, [A, np.zeros(n, dtype), np.zeros(n, dtype)], options(n))
    hiprtc_compile(s[:s.index("// host side")], options(n))
    m = re.search(r"i_\d+ < \(i_b_\d+ \+ (\d+)\); i_\d+ \+= (\d+)\)", s)
    assert (int(m[2]), int(m[1]) // int(m[2])) == (lanes, flight)


@pytest.mark.gpu
@pytest.mark.parametrize("n,avg,dtype,lanes,flight", SHAPES)
def test_sums(n, avg, dtype, lanes, flight):
    A = matrix(n, avg, dtype)
    x = np.random.default_rng(1).standard_normal(n).astype(dtype)
    y = np.full(n, -1.0, dtype)
    spmv(A, x, y, opts=options(n))
    terms = A["values"].astype(np.float64) * x[A["cols"]]
    want = np.add.reduceat(np.append(terms, 0.0), A["rows"][:-1])
    want[A["rows"][1:] == A["rows"][:-1]] = 0.0
    # rounding of up to 9001 products of size one, each sum to half a unit: far below eight units of the walk's length of 95
    assert np.abs(y - want).max() < 8 * 95 * np.finfo(dtype).eps
