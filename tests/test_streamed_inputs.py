"""Inputs of 256 MB and more that a launch reads once are read with non-temporal loads: which accesses that takes in, and
sums over whole vectors, single elements and several workgroups per row against float64."""
import numpy as np
import pytest

import parpy_amd as parpy

from kernels import max_rows, sum_rows

torch = pytest.importorskip("torch")


def twice(x, out, N):
    parpy.label('outer')
    for i in range(N):
        parpy.label('inner')
        out[i] = parpy.operators.sum(x[i, :] * x[i, :])


def again(x, out, N):
    parpy.label('outer')
    for i in range(N):
        parpy.label('inner')
        out[i] = parpy.operators.sum(x[0, :])


def scaled(x, out, N):
    parpy.label('outer')
    for i in range(N):
        parpy.label('inner')
        x[i, :] = x[i, :] * 2.0
        out[i] = 1.0


def between(x, out, first, N):
    parpy.label('outer')
    for i in range(N):
        for j in range(first[i], first[i + 1]):
            out[i] += x[j]


def picked(x, out, first, N):
    parpy.label('outer')
    for i in range(N):
        out[first[i]] = x[i]


def opts(n, m):
    return parpy.par({'outer': parpy.threads(n), 'inner': parpy.threads(m)})


def large(n, m):
    return np.zeros((n, m), dtype=np.float32)   # (untouched pages)


@pytest.mark.parametrize("f,n,m,threads,streams", [(sum_rows, 1024, 65536, 256, True), (max_rows, 1024, 65536, 64, True), (sum_rows, 7, 9600001, 8192, True),
                                                   (sum_rows, 1024, 65535, 256, False), (twice, 1024, 65536, 256, False),
                                                   (again, 1024, 65536, 256, False), (scaled, 1024, 65536, 256, False)])
def test_which_inputs_stream(f, n, m, threads, streams):
    args = [large(n, m), np.zeros(n, dtype=np.float32), n]
    f = parpy.jit(f)
    assert ("__builtin_nontemporal_load(" in parpy.print_compiled(f, args, opts(n, threads))) == streams
    plain = opts(n, threads)
    plain.opt_nontemporal = False
    assert "__builtin_nontemporal_load(" not in parpy.print_compiled(f, args, plain)


@pytest.mark.parametrize("f", [between, picked])
def test_sums_over_data_do_not_stream(f):
    args = [np.zeros(1 << 26, dtype=np.float32), np.zeros(1 << 10, dtype=np.float32), np.zeros((1 << 10) + 1, dtype=np.int64), 1 << 10]
    assert "__builtin_nontemporal_load(" not in parpy.print_compiled(parpy.jit(f), args, opts(1 << 10, 64))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tol", [(torch.float16, 4e-3), (torch.float32, 1e-5), (torch.float64, 1e-12)], ids=["f16", "f32", "f64"])
@pytest.mark.parametrize("n,m,threads", [(68, 1000003, 256), (1100, 65536, 512), (9001, 30001, 64), (3, 90000008, 8192)])
def test_streamed_sums(n, m, threads, dtype, tol):
    if dtype == torch.float16:
        m *= 2
    x = torch.rand((n, m), device="cuda", dtype=torch.float32).mul_(8192 / m if dtype == torch.float16 else 1.0).to(dtype)
    out = torch.full((2, n), -1.0, device="cuda", dtype=dtype)
    parpy.jit(sum_rows)(x, out[0], n, opts=opts(n, threads))
    parpy.jit(max_rows)(x, out[1], n, opts=opts(n, threads))
    want = torch.stack([row.double().sum() for row in x])
    assert torch.allclose(out[0].double(), want, rtol=tol, atol=0.0)
    assert torch.equal(out[1], x.max(1).values)
