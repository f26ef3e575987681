"""Reductions on more threads than a workgroup holds: shares of whole vectors with a rest, rows that start anywhere, long
shares on more and smaller workgroups, and the last workgroup reducing the partial results, call after call."""
import numpy as np
import pytest

import parpy_amd as parpy

from kernels import max_rows, min_rows, scaled_row_sums, sum_planes, sum_rows

torch = pytest.importorskip("torch")


def opts(n, m, k=1):
    return parpy.par({'outer': parpy.threads(n), 'inner': parpy.threads(m), 'N': parpy.threads(n), 'M': parpy.threads(m), 'K': parpy.threads(k)})


def test_one_launch_with_counters():
    x, out = np.zeros((3, 50003), dtype=np.float32), np.zeros(3, dtype=np.float32)
    s = parpy.print_compiled(sum_rows, [x, out, 3], opts(3, 2048))
    assert s.count("<<<") == 1 and "parpy_last_workgroup(" in s and "[3];" in s
    s = parpy.print_compiled(sum_rows, [x[:, :10000].copy(), out, 3], opts(3, 2048))
    assert s.count("<<<") == 2 and "parpy_last_workgroup(" not in s.split("extern", 1)[1]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tol", [(torch.float16, 4e-3), (torch.float32, 1e-5), (torch.float64, 1e-12)], ids=["f16", "f32", "f64"])
@pytest.mark.parametrize("threads", [2048, 8192, 32768])
def test_sums_and_extremes(threads, dtype, tol):
    for m in (threads + 1, 5 * threads - 1, 5 * threads, 5 * threads + 3, 63 * threads + 2, 64 * threads, 65 * threads + 1):
        g = torch.Generator(device="cuda").manual_seed(m)
        x = (torch.rand((3, m), generator=g, device="cuda", dtype=torch.float32) * (8192 / m if dtype == torch.float16 else 1.0)).to(dtype)
        for call in range(3):
            out = torch.full((3, 3), -1.0, device="cuda", dtype=dtype)
            for f, o in ((sum_rows, out[0]), (max_rows, out[1]), (min_rows, out[2])):
                parpy.jit(f)(x, o, 3, opts=opts(3, threads))
            assert torch.allclose(out[0].double(), x.double().sum(1), rtol=tol, atol=0.0), (m, call)
            assert torch.equal(out[1], x.max(1).values) and torch.equal(out[2], x.min(1).values), (m, call)
            x[:, -1] += 1.5   # the last element, in the rest of the last share, decides the next maximum


@pytest.mark.gpu
@pytest.mark.parametrize("k", [20003, 131073])
def test_planes_and_neighbouring_loops(k):
    x = torch.rand((3, 5, k), device="cuda") + 0.5
    out = torch.zeros((3, 5), device="cuda")
    for call in range(2):
        parpy.jit(sum_planes)(x, out, 3, 5, opts=opts(3, 5, 2048))
        assert torch.allclose(out.double(), x.double().sum(2), rtol=1e-5), call
    x, y, out = x[0].contiguous(), torch.empty((5, k), device="cuda"), torch.zeros(5, device="cuda")
    parpy.jit(scaled_row_sums)(x, y, out, 5, k, opts=opts(5, 4096))
    want = x.double() * 2.0 + 1.0
    assert torch.allclose(out.double(), want.sum(1), rtol=1e-5) and torch.allclose(y.double(), want / want.sum(1, keepdim=True), rtol=2e-5)


def test_a_split_with_small_workgroups_stays_as_it_is_named():
    x, out = np.zeros((100, 65536), dtype=np.float32), np.zeros(100, dtype=np.float32)
    s = parpy.print_compiled(sum_rows, [x, out, 100], parpy.par({'outer': parpy.threads(100), 'inner': parpy.threads(1024).tpb(128)}))
    assert s.count("<<<") == 2 and "parpy_alloc_buffer(3200)" in s


def test_a_few_long_rows_take_several_workgroups():
    # (rows, row length, element type) and whether one workgroup per row is enough
    for n, m, dtype, spread in ((1, 100000, np.float32, True), (1, 79999, np.float32, False), (30, 100001, np.float32, True), (3, 40000, np.float64, True),
                                (64, 100000, np.float32, False), (64, 131072, np.float32, True), (3, 200000, np.float16, False)):
        x, out = np.zeros((n, m), dtype=dtype), np.zeros(n, dtype=dtype)
        s = parpy.print_compiled(sum_rows, [x, out, n], opts(n, 256))
        assert s.count("<<<") == 1 and ("parpy_last_workgroup(" in s.split("extern", 1)[1]) == spread, (n, m, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tol", [(torch.int32, 0.0), (torch.float32, 1e-5), (torch.float64, 1e-12)], ids=["i32", "f32", "f64"])
@pytest.mark.parametrize("n,m", [(1, 80000), (1, 100001), (2, 1000003), (31, 163841), (64, 262147), (127, 300002)])
def test_a_few_long_rows(n, m, dtype, tol):
    x = torch.randint(1, 100, (n, m), device="cuda").to(dtype)
    for call in range(2):
        for threads in (64, 512):
            out = torch.full((3, n), -1, device="cuda", dtype=dtype)
            for f, o in ((sum_rows, out[0]), (max_rows, out[1]), (min_rows, out[2])):
                parpy.jit(f)(x, o, n, opts=opts(n, threads))
            assert torch.allclose(out[0].double(), x.double().sum(1), rtol=tol, atol=0.0), (threads, call)
            assert torch.equal(out[1], x.max(1).values) and torch.equal(out[2], x.min(1).values), (threads, call)
        x[:, -1] += 150
