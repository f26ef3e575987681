"""Sums over rows of uneven length (bounds that are data): teams of lanes per row, very long rows shared by a workgroup,
with and without columns; row counts, row lengths and column counts at the edges of what a team, a batch, a wavefront
and the queue of long rows hold.  The expectation is NumPy in float64."""
import re

import numpy as np
import pytest

import parpy_amd as parpy
from parpy_amd.compile import hiprtc_compile
from parpy_amd.operators import float32

HIP = parpy.CompileBackend.Hip


def weighted(A, x, y, z):
    parpy.label('row')
    for row in range(A["nrows"]):
        y[row] = z[row]
        parpy.label('i')
        for i in range(A["rows"][row], A["rows"][row + 1]):
            col = A["cols"][i]
            y[row] += A["values"][i] * x[col]


def columns(A, B, C, z):
    parpy.label('i')
    for i in range(A["nrows"]):
        parpy.label('j')
        for j in range(B["ncols"]):
            t = z[i] * 0.5
            parpy.label('k')
            for k in range(A["rows"][i], A["rows"][i + 1]):
                t = t + A["values"][k] * B["values"][A["cols"][k], j]
            C[i, j] = t * z[i] + 1.0


def fixed_length(x, out, N, M):
    parpy.label('i')
    for i in range(N):
        t = float32(3.0)
        for d in range(M):
            t = t + x[i, d]
        out[i] = t


def padded(A, x, perm, y):
    """Padding marked by -1, an index array that is shorter than the sums, and a test that is a load itself."""
    parpy.label('row')
    for row in range(A["nrows"]):
        y[row] = 0.0
        parpy.label('i')
        for i in range(A["rows"][row], A["rows"][row + 1]):
            y[row] += x[perm[A["cols"][i]]] if A["cols"][i] >= 0 else 0.0


def summed(A, x, y):
    parpy.label('row')
    for row in range(A["nrows"]):
        y[row] = 0.0
        parpy.label('i')
        for i in range(A["rows"][row], A["rows"][row + 1]):
            y[row] += A["values"][i] * (x[i] if i < 100 else 0.0)


def guarded(A, x, y):
    parpy.label('row')
    for row in range(A["nrows"]):
        y[row] = 0.0
        parpy.label('i')
        for i in range(A["rows"][row], A["rows"][row + 1]):
            y[row] += x[i] if i < 100 else 0.0


def ranges(first, end, x, y, n):
    """Every row with a first and a last element of its own."""
    parpy.label('row')
    for row in range(n):
        y[row] = 0.0
        parpy.label('i')
        for i in range(first[row], end[row]):
            y[row] += x[i]


def bounded(A, x, perm, y):
    parpy.label('row')
    for row in range(A["nrows"]):
        y[row] = 0.0
        parpy.label('i')
        for i in range(A["rows"][row], A["rows"][row + 1]):
            y[row] += x[A["cols"][perm[i]]] if i < 100 and perm[i] >= 0 and A["cols"][perm[i]] > 3 else 0.5


def matrix(n, m, dtype, seed):
    """Row lengths: empty, one, around a team, around the longest row a team keeps, and one that dwarfs the rest."""
    rng = np.random.default_rng(seed)
    lens = rng.choice([0, 1, 2, 7, 8, 9, 31, 32, 33], size=n)
    edge = [63, 64, 65, 127, 128, 129, 255, 256, 257, 1023, 1025, 5000]
    lens[rng.choice(n, size=len(edge), replace=False)] = edge
    rows = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    cols = rng.integers(0, m, rows[-1]).astype(np.int64)
    values = rng.standard_normal(rows[-1]).astype(dtype)
    return {"values": values, "rows": rows, "cols": cols, "nrows": n}


def row_sums(A, terms):
    """float64 sums of `terms` (one row of columns per non-zero) over the rows of A."""
    total = np.concatenate([np.zeros((1,) + terms.shape[1:]), np.cumsum(terms.astype(np.float64), axis=0)])
    return total[A["rows"][1:]] - total[A["rows"][:-1]]


def opts_for(p):
    o = parpy.par(p)
    o.backend = HIP
    return o


def test_long_rows_are_queued_for_the_workgroup():
    A = matrix(5000, 300, np.float32, 1)
    v = np.zeros(5000, dtype=np.float32)
    s = parpy.print_compiled(weighted, [A, np.zeros(300, dtype=np.float32), v, v.copy()], opts_for({"row": parpy.threads(5000)}))
    hiprtc_compile(s[:s.index("// host side")], opts_for({}))
    assert "atomicAdd(&long_count" in s and "parpy_block_reduce<parpy_op_add, 16>" in s
    B = {"values": np.zeros((300, 64), dtype=np.float32), "ncols": 64}
    s = parpy.print_compiled(columns, [A, B, np.zeros((5000, 64), dtype=np.float32), v], opts_for({"i": parpy.threads(5000), "j": parpy.threads(64)}))
    hiprtc_compile(s[:s.index("// host side")], opts_for({}))
    assert "parpy_team_sum<16, 64>" in s and "long_sums" in s


def test_loads_under_a_test_stay_under_it():
    """What a selection or a short-circuit operator may skip is not evaluated in front of the term: its index need not be one."""
    A, x, perm, y = matrix(5000, 300, np.float64, 1), np.zeros(300), np.zeros(300, dtype=np.int64), np.zeros(5000)
    for f, skipped in ((padded, ("perm",)), (bounded, ("perm", "cols"))):
        s = parpy.print_compiled(f, [A, x, perm, y], opts_for({"row": parpy.threads(5000)}))
        s = s[:s.index("// host side")]
        hiprtc_compile(s, opts_for({}))
        kernel = s[s.rindex('extern "C"'):]
        assert "parpy_block_reduce" in kernel    # (the form with teams of lanes)
        for line in kernel.splitlines():
            for name in skipped:
                at, test = re.search(rf"parpy_at\(\w*{name}_\d+,|\w*{name}_\d+\[", line), re.search(r"\?|&&", line)
                assert at is None or (test is not None and test.start() < at.start()), line


def test_loop_variables_are_narrowed_by_arrays_that_every_element_reads():
    """An array that is read under a test only says nothing about how far the rows go."""
    A, x, y = matrix(5000, 300, np.float64, 1), np.zeros(100), np.zeros(5000)

    def kernel(f):
        s = parpy.print_compiled(f, [A, x, y], opts_for({"row": parpy.threads(5000)}))
        return s[:s.index("// host side")]

    assert "int32_t end_" in kernel(summed) and "int64_t end_" in kernel(guarded)


def test_rows_without_elements_have_bounds_of_zero():
    v = np.zeros(5000, dtype=np.int64)
    for f, args in ((ranges, [v, v.copy(), np.zeros(100000), np.zeros(5000), 5000]), (guarded, [matrix(5000, 300, np.float64, 1), np.zeros(100), np.zeros(5000)])):
        s = parpy.print_compiled(f, args, opts_for({"row": parpy.threads(5000)}))
        s = s[:s.index("// host side")]
        hiprtc_compile(s, opts_for({}))
        bounds = re.findall(r"int\d+_t (?:first|end)_\d+ = (.*);", s[s.rindex('extern "C"'):])
        assert len(bounds) == 4 and all(re.search(r"any_\d+ \? (lo|hi)_\d+ : 0", b) for b in bounds), bounds


@pytest.mark.gpu
@pytest.mark.parametrize("n", [64, 1000, 20001])
def test_rows_whose_bounds_mark_that_they_are_empty(n):
    rng = np.random.default_rng(n)
    x = rng.standard_normal(5000)
    first = rng.integers(0, 4900, n)
    end = first + rng.integers(1, 100, n)
    end[:3], first[:3] = 5000, 0
    for q, (a, b) in enumerate([(2**63 - 1, 0), (2**63 - 1, -2**63), (2**32, 3), (7, 7), (2**31 + 5, 4), (100, 50), (-1, -1)]):
        first[q + 5::11], end[q + 5::11] = a, b
    y = np.full(n, np.nan)
    parpy.jit(ranges)(first, end, x, y, n, opts=opts_for({"row": parpy.threads(n)}))
    want = np.array([x[a:b].sum() if a < b else 0.0 for a, b in zip(first.tolist(), end.tolist())])
    assert np.allclose(y, want, atol=1e-10)   # (5000 terms of order one: 5000 * 5000 * 2^-53)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [65, 1025, 20001])
def test_sums_of_padded_rows(n):
    A = matrix(n, 300, np.float64, n)
    rng = np.random.default_rng(n + 2)
    A["cols"][rng.random(len(A["cols"])) < 0.3] = -1
    x, perm, y = rng.standard_normal(300), rng.permutation(300).astype(np.int64), np.full(n, np.nan)
    parpy.jit(padded)(A, x, perm, y, opts=opts_for({"row": parpy.threads(n)}))
    want = row_sums(A, np.where(A["cols"] >= 0, x[perm[A["cols"]]], 0.0))
    # (partial sums of the whole vector, at most 400000 terms of order one: 400000 * 2^-53 * 600 at the very most)
    assert np.allclose(y, want, atol=1e-7)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("n", [64, 65, 1000, 1025, 20001])
def test_sums_of_uneven_rows(n, dtype):
    A = matrix(n, 300, dtype, n)
    rng = np.random.default_rng(n + 1)
    x, z, y = rng.standard_normal(300).astype(dtype), rng.standard_normal(n).astype(dtype), np.full(n, np.nan, dtype=dtype)
    parpy.jit(weighted)(A, x, y, z, opts=opts_for({"row": parpy.threads(n)}))
    want = z + row_sums(A, A["values"].astype(np.float64) * x[A["cols"]])
    assert np.allclose(y, want, atol=1e-3 if dtype == np.float32 else 1e-9)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("n,cols", [(64, 1), (65, 3), (100, 32), (1000, 100), (300, 101), (129, 256), (200, 258), (70, 513), (64, 1024)])
def test_sums_of_uneven_rows_with_columns(n, cols, dtype):
    A = matrix(n, 50, dtype, n)
    rng = np.random.default_rng(cols)
    B, z, C = rng.standard_normal((50, cols)).astype(dtype), rng.standard_normal(n).astype(dtype), np.full((n, cols), np.nan, dtype=dtype)
    parpy.jit(columns)(A, {"values": B, "ncols": cols}, C, z, opts=opts_for({"i": parpy.threads(n), "j": parpy.threads(cols)}))
    want = (0.5 * z[:, None] + row_sums(A, A["values"].astype(np.float64)[:, None] * B[A["cols"]])) * z[:, None] + 1.0
    assert np.allclose(C, want, atol=2e-3 if dtype == np.float32 else 1e-9)


@pytest.mark.gpu
def test_start_value_of_a_shared_sum_counts_once():
    x = np.random.default_rng(3).standard_normal((300, 132)).astype(np.float32)
    out = np.zeros(300, dtype=np.float32)
    parpy.jit(fixed_length)(x, out, 300, 132, opts=opts_for({'i': parpy.threads(300)}))
    assert np.allclose(out, 3.0 + x.astype(np.float64).sum(1), atol=1e-4)


def outliers(n, dtype, long, seed):
    """Short rows and, at the places given, rows around and beyond the length that workgroups of their own look for."""
    rng = np.random.default_rng(seed)
    lens = rng.integers(0, 8, size=n)
    for row, length in long.items():
        lens[row] = length
    rows = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    return {"values": rng.standard_normal(rows[-1]).astype(dtype), "rows": rows, "cols": rng.integers(0, 300, rows[-1]).astype(np.int64), "nrows": n}


LONG = {0: 20000, 1: 1024, 2: 1025, 3: 1026, 77: 256, 78: 257, 79: 64, 80: 65, 81: 258, 5000: 4097, 5001: 4096, 5002: 4095, 60001: 12345, -2: 3000, -1: 9999}


def test_outliers_are_looked_for_where_not_all_rows_run_at_once():
    for n, found in ((8192, False), (8193, True)):   # (a wavefront per row)
        A, z = outliers(n, np.float32, {}, 1), np.zeros(n, dtype=np.float32)
        B = {"values": np.zeros((300, 33), dtype=np.float32), "ncols": 33}
        s = parpy.print_compiled(columns, [A, B, np.zeros((n, 33), dtype=np.float32), z], opts_for({"i": parpy.threads(n), "j": parpy.threads(33)}))
        assert ("slice_" in s) == found
        hiprtc_compile(s[:s.index("// host side")], opts_for({}))


@pytest.mark.gpu
@pytest.mark.parametrize("n,cols", [(70000, 33), (8193, 33), (9001, 256), (17000, 128)])
def test_outliers_with_columns(n, cols):
    for long in ({k if k < n else n - 5: min(v, 5000) for k, v in LONG.items()}, {}, {n // 2: 20000}, {r: 300 for r in range(1000, 1200)}):
        A = outliers(n, np.float32, long, n)
        rng = np.random.default_rng(cols)
        B, z, C = rng.standard_normal((300, cols)).astype(np.float32), rng.standard_normal(n).astype(np.float32), np.full((n, cols), np.nan, dtype=np.float32)
        parpy.jit(columns)(A, {"values": B, "ncols": cols}, C, z, opts=opts_for({"i": parpy.threads(n), "j": parpy.threads(cols)}))
        want = (0.5 * z[:, None] + row_sums(A, A["values"].astype(np.float64)[:, None] * B[A["cols"]])) * z[:, None] + 1.0
        # (a sum of 20000 products of order one is off by 20000 * 2^-24 * 100 at the very most: 0.1; 5e-3 is what their random signs leave)
        assert np.allclose(C, want, atol=5e-3)
