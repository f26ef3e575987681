"""Sums over sparse rows: rows that a workgroup shares, around its batches of eight elements a thread; few rows, whose lanes follow
the average row; workgroups in front of launches that fill the device."""
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


# rows, average, type, lanes of a row, workgroups in front
SHAPES = [(1000, 47, np.float32, 8, 0), (1000, 48, np.float64, 32, 0), (900, 100, np.float32, 64, 0), (65, 300, np.float64, 64, 0),
          (16000, 60, np.float64, 32, 256), (8000, 150, np.float64, 64, 256), (14400, 60, np.float64, 32, 256), (16000, 60, np.float32, 32, 0),
          (14100, 60, np.float64, 32, 71), (5000, 100, np.float32, 64, 199), (1100, 100, np.float64, 64, 68)]


@pytest.mark.parametrize("n,avg,dtype,lanes,in_front", SHAPES)
def test_lanes_and_workgroups_in_front(n, avg, dtype, lanes, in_front):
    A = {"values": np.zeros(n * avg, dtype), "rows": np.arange(n + 1) * avg, "cols": np.zeros(n * avg, np.int64), "nrows": n}
    s = parpy.print_compiled(spmv, [A, np.zeros(n, dtype), np.zeros(n, dtype)], options(n))
    hiprtc_compile(s[:s.index("// host side")], options(n))
    m = re.search(r"if \(blockIdx.x >= (\d+)\) return;", s)
    assert (int(m[1]) if m else 0) == in_front
    steps = [(int(b), int(d)) for b, d in re.findall(r"i_\d+ < \(i_b_\d+ \+ (\d+)\); i_\d+ \+= (\d+)\)", s)]
    tpb = int(re.search(r"__launch_bounds__\((\d+)\)", s)[1])
    assert steps[0][1] == lanes and steps[1:] == [(8 * tpb, tpb), (4 * tpb, tpb)]


@pytest.mark.gpu
@pytest.mark.parametrize("n,avg,dtype,lanes,in_front", SHAPES)
def test_sums(n, avg, dtype, lanes, in_front):
    rng = np.random.default_rng(n)
    lengths = rng.integers(0, 2 * avg - 1, n)
    edges = [0, 1, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025, 2047, 2048, 2049, 4095, 4096, 4097, 8191, 8192, 8193, 12289, 16384, 18433]
    lengths[rng.choice(n, len(edges), replace=False)] = edges
    lengths[[0, n - 1]] = 4097, 8192
    rows = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    A = {"values": rng.standard_normal(rows[-1]).astype(dtype), "rows": rows, "cols": rng.integers(0, n, rows[-1]), "nrows": n}
    x = rng.standard_normal(n).astype(dtype)
    y = np.full(n, -1.0, dtype)
    spmv(A, x, y, opts=options(n))
    terms = A["values"].astype(np.float64) * x[A["cols"]]
    want = np.add.reduceat(np.append(terms, 0.0), rows[:-1])
    want[rows[1:] == rows[:-1]] = 0.0
    # rounding of up to 18433 products of size one, each sum to half a unit: far below eight units of the walk's length of 136
    assert np.abs(y - want).max() < 8 * 136 * np.finfo(dtype).eps
