"""Transposed copies of tables: tiles that the table does not fill, rows that start on cache lines, and copies that fit the fixed
memory of a run that may allocate nothing only without that."""
import re

import numpy as np
import pytest
import torch

import parpy_amd as parpy
from parpy_amd import workloads as W
from parpy_amd.compile import hiprtc_compile

# rows of the table, columns (its copy's rows), element type, elements between the copy's rows
SHAPES = [(255, 300, "float32", 255), (257, 300, "float32", 288), (129, 65, "float64", 144), (128, 64, "float64", 128), (333, 63, "float32", 333),
          (1023, 129, "float32", 1024), (31, 4099, "float64", 31), (64, 1000, "float32", 64), (1025, 1100, "float64", 1040)]


def options(nnz):
    o = parpy.par({"nnz": parpy.threads(nnz).tpb(256)})
    o.backend = parpy.CompileBackend.Hip
    return o


def listing(n, k, nnz, dtype):
    z = lambda *shape: np.zeros(shape, dtype)
    C = {"rows": np.zeros(nnz, np.int64), "cols": np.zeros(nnz, np.int64), "values": z(nnz), "nnz": nnz}
    return parpy.print_compiled(W.sddmm_coo, [z(70, k), z(k, n), C, z(nnz), np.dtype(dtype).type(1.5), np.dtype(dtype).type(2.0)], options(nnz))


def bytes_copied(s):
    return int(re.search(r"B_T_\d+ = \(\w+\*\)parpy_alloc_buffer\((\d+)\)", s).group(1))


@pytest.mark.parametrize("k,n,dtype,pitch", SHAPES)
def test_rows_of_a_copy(k, n, dtype, pitch):
    s = listing(n, k, 900, dtype)
    hiprtc_compile(s[:s.index("// host side")], options(900))
    assert bytes_copied(s) == pitch * n * np.dtype(dtype).itemsize


def test_copies_that_fit_stay_so():
    # 16 MiB: with whole lines 15.3 of them would be above seven eighths, and 17.6 above all; a copy that never fitted has lines
    for n, k, pitch in ((3800, 1025, 1025), (4050, 1025, 1025), (4200, 1025, 1056), (3400, 1025, 1056)):
        assert bytes_copied(listing(n, k, 900, "float32")) == n * pitch * 4


@pytest.mark.gpu
@pytest.mark.parametrize("k,n,dtype,pitch", SHAPES)
def test_products_out_of_a_copy(k, n, dtype, pitch):
    rng = np.random.default_rng(k)
    A, B = rng.standard_normal((70, k), np.float32).astype(dtype), rng.standard_normal((k, n), np.float32).astype(dtype)
    nnz = 2 * n + 3
    rows, cols = rng.integers(0, 70, nnz), np.concatenate([np.arange(n), np.arange(n)[::-1], [0, n - 1, n // 2]])
    vals = rng.standard_normal(nnz).astype(dtype)
    dev = [torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in (A, B, rows, cols, vals)]
    D = torch.full((nnz,), -7.0, dtype=dev[0].dtype, device="cuda")
    one = np.dtype(dtype).type
    W.sddmm_coo(dev[0], dev[1], {"rows": dev[2], "cols": dev[3], "values": dev[4], "nnz": nnz}, D, one(1.5), one(2.0), opts=options(nnz))
    x, y = A[rows].astype(np.float64), B.T[cols].astype(np.float64)
    want = 1.5 * (x * y).sum(1) + 2.0 * vals.astype(np.float64)
    # at most k additions and products, each rounded once
    bound = (1.5 * np.abs(x * y).sum(1) * (k + 3) + 4 * np.abs(vals) + 3 * np.abs(want)) * np.finfo(dtype).eps / 2
    assert (np.abs(D.cpu().numpy() - want) <= bound).all()
