"""Products of rows that memory selects out of large tables, cut into slabs along the rows: rows that are no whole number of
slabs, pieces or vectors, more slabs than dies, a number of products that no workgroup divides, and no room for the parts."""
import re

import numpy as np
import pytest
import torch

import parpy_amd as parpy
from parpy_amd import workloads as W
from parpy_amd.compile import hiprtc_compile

# rows of the tables, their length, products, element type, slabs that the rule chooses (33 pieces of 128 bytes: no eight slabs of whole pieces)
SHAPES = [(2400, 1024, 37013, "float32", 2), (5200, 1024, 25000, "float32", 8), (5300, 1024, 13001, "float64", 16), (6000, 777, 33003, "float32", 4),
          (3100, 780, 33000, "float64", 4), (9000, 331, 39001, "float64", 4), (5300, 1021, 25011, "float32", 8), (5300, 1050, 25011, "float32", 4), (2400, 1024, 36000, "float32", 1),
          (2200, 1024, 37013, "float32", 1), (17000, 200, 130000, "float32", 1), (12000, 264, 100003, "float32", 2)]


def operands(n, k, nnz, dtype):
    rng = np.random.default_rng(n + k)
    A, B = rng.standard_normal((n, k), np.float32).astype(dtype), rng.standard_normal((k, n), np.float32).astype(dtype)
    rows, cols = rng.integers(0, n, nnz), rng.integers(0, n, nnz)
    rows[: nnz // 2].sort()
    return A, B, rows, cols, rng.standard_normal(nnz).astype(dtype)


def options(nnz, tpb=256, **flags):
    o = parpy.par({"nnz": parpy.threads(nnz).tpb(tpb)})
    o.backend = parpy.CompileBackend.Hip
    for key, value in flags.items():
        setattr(o, key, value)
    return o


def listing(n, k, nnz, dtype, to=lambda x: x, **flags):
    z = lambda *shape: np.zeros(shape, dtype)
    C = {"rows": np.zeros(nnz, np.int64), "cols": np.zeros(nnz, np.int64), "values": z(nnz), "nnz": nnz}
    return parpy.print_compiled(W.sddmm_coo, [z(n, k), z(k, n), C, z(nnz), np.dtype(dtype).type(1.5), np.dtype(dtype).type(2.0)], options(nnz, **flags))


def slabs_in(text):
    parts = re.search(r"(float|double)\* t_parts_\d+ = \(\w+\*\)parpy_alloc_buffer\((\d+)\)", text)
    products = re.search(r"t_parts_\d+\[\(\(slab_\d+ \* (\d+)\)", text)
    return int(parts.group(2)) // ((4 if parts.group(1) == "float" else 8) * int(products.group(1))) if parts else 1


@pytest.mark.parametrize("n,k,nnz,dtype,slabs", SHAPES)
def test_slabs_of_a_shape(n, k, nnz, dtype, slabs):
    s = listing(n, k, nnz, dtype)
    hiprtc_compile(s[:s.index("// host side")], options(nnz))
    assert slabs_in(s) == slabs
    # every element of a row belongs to one slab: the first elements and the lengths of all but the last are the same
    if slabs > 1:
        es = np.dtype(dtype).itemsize
        vec, chunks = 16 // es, -(-k * es // 128)
        width = -(-chunks // slabs) * 8
        assert re.search(rf"\(slab_\d+ \* {width}\)", s) and (slabs - 1) * width * vec < k


def test_parts_beyond_what_a_plan_keeps():
    # 16 * 10^6 products in eight slabs: parts of 488 MiB, beside a copy of 391 MiB and one of 781 (zeros that are never touched)
    assert slabs_in(listing(100000, 1024, 16000000, "float32")) == 8
    assert slabs_in(listing(200000, 1024, 16000000, "float32")) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("tpb", [256, 64])
@pytest.mark.parametrize("n,k,nnz,dtype,slabs", SHAPES)
def test_products_in_slabs(n, k, nnz, dtype, slabs, tpb):
    A, B, rows, cols, vals = operands(n, k, nnz, dtype)
    dev = [torch.from_numpy(x).cuda() for x in (A, B, rows, cols, vals)]
    C = {"rows": dev[2], "cols": dev[3], "values": dev[4], "nnz": nnz}
    one = np.dtype(dtype).type
    D = [torch.full((nnz,), -7.0, dtype=dev[0].dtype, device="cuda") for _ in range(2)]
    W.sddmm_coo(dev[0], dev[1], C, D[0], one(1.5), one(2.0), opts=options(nnz, tpb))
    W.sddmm_coo(dev[0], dev[1], C, D[1], one(1.5), one(2.0), opts=options(nnz, tpb, opt_lane_split=False))
    Bt = np.ascontiguousarray(B.T)
    want = np.empty(nnz)
    size = np.empty(nnz)
    for i in range(0, nnz, 8192):
        x, y = A[rows[i:i + 8192]].astype(np.float64), Bt[cols[i:i + 8192]].astype(np.float64)
        want[i:i + 8192] = np.einsum("ij,ij->i", x, y)
        size[i:i + 8192] = np.einsum("ij,ij->i", np.abs(x), np.abs(y))
    want = 1.5 * want + 2.0 * vals.astype(np.float64)
    # a sum of at most a lane's k / 8 products, eight lanes' and the slabs', each addition and product rounded once
    eps = np.finfo(dtype).eps / 2
    bound = (1.5 * size * (k / 8 + 3 + 64) + 4 * np.abs(vals) + np.abs(want) * 3) * eps
    err = [np.abs(d.cpu().numpy().astype(np.float64) - want) for d in D]
    assert (err[0] <= bound).all()
    # and no less exact than one thread's sum over the whole row
    assert np.sqrt((err[0] ** 2).mean()) <= np.sqrt((err[1] ** 2).mean())


@pytest.mark.gpu
@pytest.mark.parametrize("n,k,nnz,dtype", [(5300, 1024, 25011, "float32"), (6000, 777, 33003, "float32"), (9000, 331, 39001, "float64"), (5300, 1021, 25011, "float32")])
def test_infinities_where_slabs_meet(n, k, nnz, dtype):
    """Elements that another slab's last vector holds as well, or that stand in front of a moved one, count once and in their own row."""
    A, B, rows, cols, vals = operands(n, k, nnz, dtype)
    A[:] = B[:] = 1.0
    at = [0, 1, k // 8, k // 4 - 1, k // 4, k // 2, k - 5, k - 4, k - 3, k - 2, k - 1]
    for q, d in enumerate(at):
        A[10 * q, d], A[10 * q + 1, d], B[d, 10 * q] = np.inf, np.nan, 3.0
    dev = [torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in (A, B, rows, cols, vals)]
    D = torch.full((nnz,), -7.0, dtype=dev[0].dtype, device="cuda")
    one = np.dtype(dtype).type
    W.sddmm_coo(dev[0], dev[1], {"rows": dev[2], "cols": dev[3], "values": torch.zeros_like(dev[4]), "nnz": nnz}, D, one(1.0), one(0.0), opts=options(nnz))
    clean = np.where(np.isfinite(A), A, 0.0).sum(1)
    want = np.where(np.isnan(A).any(1)[rows], np.nan, np.where(np.isinf(A).any(1)[rows], np.inf, clean[rows]))
    for q, d in enumerate(at):
        want = want + np.where((cols == 10 * q) & np.isfinite(want), 2.0 * A[rows, d], 0.0)
    assert np.array_equal(D.cpu().numpy(), want, equal_nan=True)    # (whole numbers below 2^11)


@pytest.mark.gpu
def test_parts_that_find_no_room():
    """A run that may allocate nothing has 16 MiB: the copy of a table takes 9.8 MB of them, the parts 0.3 or 8.4 more."""
    n, k = 2400, 1024
    for nnz, launches in ((37013, 3), (1050000, 2)):
        A, B, rows, cols, vals = operands(n, k, nnz, "float32")
        dev = [torch.from_numpy(x).cuda() for x in (A, B, rows, cols, vals)]
        C = {"rows": dev[2], "cols": dev[3], "values": dev[4], "nnz": nnz}
        D, got = (torch.full((nnz,), -7.0, device="cuda") for _ in range(2))
        args = [dev[0], dev[1], C, D, np.float32(1.5), np.float32(2.0)]
        assert f"parpy_temporaries_fit({2 * nnz * 4})" in listing(n, k, nnz, "float32")
        W.sddmm_coo(*args, opts=options(nnz))
        parpy.sync(parpy.CompileBackend.Hip)
        o = parpy.backend._resolve_backend(options(nnz), True)
        run = parpy._compile_function(parpy._ir_asts[W.sddmm_coo], parpy.validate.check_arguments(args, o, True), o)
        assert run.launch_count() == 3
        run.run_noalloc([t.data_ptr() for t in (dev[0], dev[1], dev[3], dev[2], dev[4], got)])
        torch.cuda.synchronize()
        assert run.launch_count() == launches
        # two parts of 512 products or one sum of 1024, eight lanes each: both within what rounding allows, and the same if cut alike
        assert (got - D).abs().max().item() <= (2 * 1.5 * 1024 * 4 * (1024 / 8 + 64) * 2.0 ** -24 if launches == 2 else 0.0)


@pytest.mark.gpu
def test_products_in_slabs_captured():
    """Recorded into a graph and replayed, with other values between the replays."""
    n, k, nnz = 2400, 1024, 37013
    A, B, rows, cols, vals = operands(n, k, nnz, "float32")
    dev = [torch.from_numpy(x).cuda() for x in (A, B, rows, cols, vals)]
    C = {"rows": dev[2], "cols": dev[3], "values": dev[4], "nnz": nnz}
    D, E = (torch.full((nnz,), -7.0, device="cuda") for _ in range(2))
    for turn in range(6):
        dev[0].mul_(1.25)
        W.sddmm_coo(dev[0], dev[1], C, D, np.float32(1.5), np.float32(2.0), opts=options(nnz, use_cuda_graphs=True))
        W.sddmm_coo(dev[0], dev[1], C, E, np.float32(1.5), np.float32(2.0), opts=options(nnz))
        torch.cuda.synchronize()
        assert torch.equal(D, E), turn
