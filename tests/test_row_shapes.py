"""Reductions and softmax over rows of all lengths, element types and thread counts against float64: rows that share a
workgroup (a wavefront each, the last workgroup not full), rows cut to fewer threads, vectors of 2-, 4- and 8-byte
elements whose last one is partial, peeled last trips; quotients of halves."""
import numpy as np
import pytest

import parpy_amd as parpy
from parpy_amd import workloads as W

torch = pytest.importorskip("torch")


def centred(x, out, N, M):
    """In place, with a reduction between two element loops: an element handled twice would show."""
    parpy.label('N')
    for i in range(N):
        parpy.label('M')
        s = parpy.operators.sum(x[i, :])
        parpy.label('M')
        x[i, :] = x[i, :] * 2.0 - s
        parpy.label('M')
        out[i] = parpy.operators.max(x[i, :])


def opts(n, m):
    return parpy.par({'N': parpy.threads(n), 'M': parpy.threads(m), 'outer': parpy.threads(n), 'inner': parpy.threads(m)})


def test_short_rows_share_a_workgroup():
    x = np.zeros((9001, 200), dtype=np.float32)
    s = parpy.print_compiled(W.softmax, [x, 9001, 200, x.copy()], opts(9001, 256))
    assert "<<<dim3(1, 2251, 1), dim3(64, 4, 1)" in s and "parpy_wave_reduce<parpy_op_max>" in s and "< 9001) {" in s
    s = parpy.print_compiled(W.softmax, [x[:100], 100, 200, x[:100].copy()], opts(100, 256))
    assert "<<<dim3(1, 100, 1), dim3(256, 1, 1)" in s


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tol", [(torch.float16, 4e-3), (torch.float32, 1e-5), (torch.float64, 1e-12)], ids=["f16", "f32", "f64"])
@pytest.mark.parametrize("n,threads", [(5, 256), (4099, 64), (2049, 256), (5003, 128)])
def test_rows_of_all_lengths(n, threads, dtype, tol):
    for m in (1, 7, 63, 64, 65, 127, 128, 129, 250, 511, 513, 1000, 1777, 2047):
        g = torch.Generator(device="cuda").manual_seed(m)
        x = torch.randn((n, m), generator=g, device="cuda", dtype=torch.float32).to(dtype)
        out = torch.full_like(x, -1.0)
        W.softmax(x, n, m, out, opts=opts(n, threads))
        e = torch.exp(x.double() - x.double().max(1, keepdim=True).values)
        want = e / e.sum(1, keepdim=True)
        assert ((out.double() - want).norm() / want.norm()) < tol, (n, m)
        sums = torch.full((n,), -1.0, device="cuda", dtype=dtype)
        W.sum_rows(x, sums, n, opts=opts(n, threads))
        assert torch.allclose(sums.double(), x.double().sum(1), rtol=tol, atol=tol * 30), (n, m)
        y = x.clone()
        top = torch.full((n,), -1.0, device="cuda", dtype=dtype)
        parpy_centred(y, top, n, m, opts=opts(n, threads))
        want = x.double() * 2.0 - x.double().sum(1, keepdim=True)
        assert torch.allclose(y.double(), want, rtol=tol, atol=tol * 60), (n, m)
        assert torch.equal(top, y.max(1).values), (n, m)


parpy_centred = parpy.jit(centred)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tol", [(torch.float16, 4e-3), (torch.float32, 1e-5), (torch.float64, 1e-12)], ids=["f16", "f32", "f64"])
def test_few_long_rows_get_more_threads(dtype, tol):
    for n, m, threads in ((1, 8191, 64), (3, 20003, 64), (7, 4100, 128), (500, 33000, 128)):
        x = torch.rand((n, m), device="cuda", dtype=torch.float32).to(dtype)
        y = torch.empty_like(x)
        sums = torch.zeros(n, device="cuda", dtype=dtype)
        W.sum_rows(x, sums, n, opts=opts(n, threads))
        assert torch.allclose(sums.double(), x.double().sum(1), rtol=tol), (n, m)
        W.softmax(x, n, m, y, opts=opts(n, threads))
        e = torch.exp(x.double() - x.double().max(1, keepdim=True).values)
        want = e / e.sum(1, keepdim=True)
        assert ((y.double() - want).norm() / want.norm()) < tol, (n, m)


@parpy.jit
def quotient(a, b, out):
    parpy.label('N')
    out[:] = a[:] / b[:]


@pytest.mark.gpu
def test_quotients_of_halves_are_correctly_rounded():
    """Every numerator with a spread of denominators (all significands, large, small and subnormal ones, zeros,
    infinities, NaN) against the quotient in double precision rounded once."""
    every = torch.arange(1 << 16, dtype=torch.int32).to(torch.int16).view(torch.float16)
    denominators = torch.cat([every[0x3C00:0x4000], every[torch.tensor([0x0001, 0x0003, 0x03FF, 0x0400, 0x1234, 0x7BFF, 0x7C00, 0x7E00, 0x0000, 0x8000, 0xC123, 0xFC00])]])
    a = every.cuda().repeat(64).contiguous()
    for k in range(0, denominators.numel(), 64):
        d = denominators[k:k + 64]
        d = torch.cat([d, d[:1].expand(64 - d.numel())])
        b = d.cuda().repeat_interleave(1 << 16).contiguous()
        out = torch.empty_like(a)
        quotient(a, b, out, opts=parpy.par({'N': parpy.threads(a.numel())}))
        want = (a.double() / b.double()).to(torch.float16)
        same = (out.view(torch.int16) == want.view(torch.int16)) | (out.isnan() & want.isnan())
        assert bool(same.all()), (a[~same][:4], b[~same][:4], out[~same][:4], want[~same][:4])
