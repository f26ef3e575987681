"""Sums that eight lanes share, over lengths that are no whole number of vectors or rounds of the group: sampled products
against float64, through a transposed copy whose edge tiles are partial."""
import numpy as np
import pytest

import parpy_amd as parpy
from parpy_amd import workloads as W

torch = pytest.importorskip("torch")

LENGTHS = (16, 31, 32, 33, 35, 47, 63, 64, 65, 66, 95, 97, 127, 129, 777)


def opts(nnz):
    return parpy.par({'nnz': parpy.threads(nnz).tpb(256)})


def test_which_lengths_are_shared():
    for dtype, least in ((np.float32, 32), (np.float64, 16)):
        for k in (15, 16, 31, 32, 33, 777):
            C = {"cols": np.zeros(640, np.int64), "rows": np.zeros(640, np.int64), "values": np.zeros(640, dtype), "nnz": 640}
            s = parpy.print_compiled(W.sddmm_coo, [np.zeros((70, k), dtype), np.zeros((k, 70), dtype), C, np.zeros(640, dtype), 1.0, 0.5], opts(640))
            assert ("= parpy_sum8(" in s) == (k >= least), (dtype, k)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.float64, 1e-12)], ids=["f32", "f64"])
@pytest.mark.parametrize("n,nnz", [(70, 640), (257, 5001)])
def test_sampled_products(n, nnz, dtype, tol):
    for k in LENGTHS:
        g = torch.Generator(device="cuda").manual_seed(k)
        A = torch.randn((n, k), generator=g, device="cuda", dtype=dtype)
        B = torch.randn((k, n), generator=g, device="cuda", dtype=dtype)
        rows = torch.randint(0, n, (nnz,), generator=g, device="cuda")
        cols = torch.randint(0, n, (nnz,), generator=g, device="cuda")
        rows[-1], cols[-1] = n - 1, n - 1
        values = torch.randn(nnz, generator=g, device="cuda", dtype=dtype)
        D = torch.zeros_like(values)
        W.sddmm_coo(A, B, {"cols": cols, "rows": rows, "values": values, "nnz": nnz}, D, 1.0, 0.5, opts=opts(nnz))
        want = (A.double()[rows] * B.double().T[cols]).sum(1) + 0.5 * values.double()
        assert ((D.double() - want).norm() / want.norm()) < tol, k


def test_which_products_are_paired():
    for n, nnz, k, dtype, paired in ((8192, 140000, 128, np.float32, True), (8192, 131072, 128, np.float32, False), (8320, 140000, 128, np.float32, False),
                                     (900, 140000, 256, np.float32, False), (900, 140001, 64, np.float64, True), (900, 140000, 100, np.float32, False)):
        C = {"cols": np.zeros(nnz, np.int64), "rows": np.zeros(nnz, np.int64), "values": np.zeros(nnz, dtype), "nnz": nnz}
        s = parpy.print_compiled(W.sddmm_coo, [np.zeros((n, k), dtype), np.zeros((k, n), dtype), C, np.zeros(nnz, dtype), 1.0, 0.5], opts(nnz))
        assert ("_pair_" in s) == paired, (n, nnz, k, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,lengths,tol", [(torch.float32, (32, 64, 96, 128), 1e-5), (torch.float64, (16, 48, 64), 1e-12)], ids=["f32", "f64"])
@pytest.mark.parametrize("nnz", [131073, 140000, 140001])
@pytest.mark.parametrize("order", ["rows", "runs of one", "none", "one row"])
def test_pairs_of_products(nnz, order, dtype, lengths, tol):
    n = 301
    for k in lengths:
        g = torch.Generator(device="cuda").manual_seed(k)
        A = torch.randn((n, k), generator=g, device="cuda", dtype=dtype)
        B = torch.randn((k, n), generator=g, device="cuda", dtype=dtype)
        rows = torch.randint(0, n, (nnz,), generator=g, device="cuda")
        rows = {"rows": rows.sort().values, "none": rows, "runs of one": torch.arange(nnz, device="cuda") % n, "one row": torch.full_like(rows, n - 1)}[order]
        cols = torch.randint(0, n, (nnz,), generator=g, device="cuda")
        values = torch.randn(nnz, generator=g, device="cuda", dtype=dtype)
        D = torch.full((nnz + 1,), 7.0, device="cuda", dtype=dtype)
        W.sddmm_coo(A, B, {"cols": cols, "rows": rows, "values": values, "nnz": nnz}, D[:nnz], 1.0, 0.5, opts=opts(nnz))
        want = (A.double()[rows] * B.double().T[cols]).sum(1) + 0.5 * values.double()
        assert ((D[:nnz].double() - want).norm() / want.norm()) < tol and D[nnz] == 7.0, k
