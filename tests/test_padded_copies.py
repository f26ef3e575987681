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


@parpy.jit
def gathered(X, Y, Z, cols, out, n, k):
    parpy.label('nnz')
    for i in range(n):
        c = cols[i]
        t = 0.0
        for d in range(k):
            t += X[d, c] * Y[d, c]
        out[i] = t
    parpy.label('nnz')
    for i in range(n):
        c = cols[i]
        t = 0.0
        for d in range(k):
            t += Z[d, c]
        out[i] += t


def plan_of(k, x, y, z):
    f = lambda n: np.zeros((k, n), np.float32)
    return parpy.print_compiled(gathered, [f(x), f(y), f(z), np.zeros(900, np.int64), np.zeros(900, np.float32), 900, k], options(900))


def most_at_once(s):
    """Bytes in use at most where only the last temporary gives its place back before the run ends, and all bytes."""
    live, top, most, total = [], 0, 0, 0
    for name, size, freed in re.findall(r"(\w+) = \(\w+\*\)parpy_alloc_buffer\((\d+)\)|parpy_free_buffer\((\w+)\)", s):
        if freed and live[-1][0] == freed:
            top = live.pop()[1]
        elif not freed:
            live.append((name, top))
            top = -(-top // 256) * 256 + int(size)
            most, total = max(most, top), total + int(size)
    return most, total


# columns of two tables that one launch copies and of the next launch's; what is added to their rows of 260 elements
@pytest.mark.parametrize("x,y,z,added", [(5000, 5000, 9900, 28), (7800, 7700, 5000, (0, 28)), (5000, 5000, 5000, 28), (420000, 420000, 150000, 0)])
def test_copies_of_several_tables(x, y, z, added):
    s, k = plan_of(260, x, y, z), 260
    sizes = {m[0]: int(m[1]) for m in re.findall(r"([XYZ])_T_\d+ = \(float\*\)parpy_alloc_buffer\((\d+)\)", s)}
    first, second = added if isinstance(added, tuple) else (added, added)
    assert sizes == {"X": 4 * x * (k + first), "Y": 4 * y * (k + first), "Z": 4 * z * (k + second)}
    most, total = most_at_once(s)
    if 4 * k * (x + y) + 512 <= 16 << 20 and 4 * k * z <= 16 << 20:
        assert most <= 16 << 20     # what a run that allocates nothing has
    if 4 * k * (x + y + z) <= 1 << 30:
        assert total <= 1 << 30     # what a plan keeps for captured runs


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
