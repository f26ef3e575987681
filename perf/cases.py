"""The measured workloads of this package: what programs that use it run, over the range of sizes they run it at.

`listed()` names twelve calls, `draw()` makes more of the same families, `prepare()` builds what a program holds
before the call (seeded inputs on the GPU and the arrays for the results), `run()` is the call itself, written as the
package's own examples write it: a jitted function, device tensors, and `opts=parpy.par({...})` built where the call
stands.  Families:

  rows      row sums of a matrix, from ten short rows to ten rows of 10^7 elements on several workgroups per row
  softmax   the four-statement row softmax, single, double and half precision, row lengths that fill no whole vector
  sddmm     sampled dense-dense products on a COO or CSR mask
  spmv      CSR matrix times vector, rows of uneven length
  spmm      CSR matrix times a dense matrix
  jacobi    a three-point stencil swept back and forth, time loop on the host
  hmm       HMM forward pass, synthetic 4^k-state model, in the three statements of `parpy_amd.workloads`
  hmm16     HMM forward pass of the 16-layer nanopore model, unchanged user code or in scaled linear space
"""
import math

import torch

import parpy_amd as parpy
from parpy_amd import workloads as W

DTYPES = {"f16": torch.float16, "f32": torch.float32, "f64": torch.float64}
SIZEOF = {"f16": 2, "f32": 4, "f64": 8}
OBSERVATIONS = 101


# ---------------------------------------------------------------- user programs that the package's workloads do not hold
@parpy.jit
def spmv(A, x, y):
    parpy.label('row')
    for row in range(A["nrows"]):
        y[row] = 0.0
        parpy.label('i')
        for i in range(A["rows"][row], A["rows"][row + 1]):
            y[row] += A["values"][i] * x[A["cols"][i]]


@parpy.jit
def spmm(A, B, C):
    parpy.label('i')
    for i in range(A["nrows"]):
        parpy.label('j')
        for j in range(B["ncols"]):
            C[i, j] = 0.0
            parpy.label('aidx')
            for aidx in range(A["rows"][i], A["rows"][i + 1]):
                C[i, j] += A["values"][aidx] * B["values"][A["cols"][aidx], j]


@parpy.jit
def jacobi(nsteps, A, B):
    for t in range(1, nsteps):
        parpy.label('N')
        B[1:-1] = (A[:-2] + A[1:-1] + A[2:]) / 3.0
        parpy.label('N')
        A[1:-1] = (B[:-2] + B[1:-1] + B[2:]) / 3.0


# ---------------------------------------------------------------- cases
def listed():
    return [
        # the smallest call: ten short rows, one workgroup each; what a call costs at all
        {"name": "rows 10x1000", "family": "rows", "n": 10, "m": 1000, "dtype": "f32", "threads": 1024},
        # the motivating example of the language: few huge rows, 32 workgroups per row and a second reduction stage
        {"name": "rows 10x10000000", "family": "rows", "n": 10, "m": 10000000, "dtype": "f32", "threads": 32768},
        # the row-sum benchmark
        {"name": "rows 1024x65536", "family": "rows", "n": 1024, "m": 65536, "dtype": "f32", "threads": 256},
        # the softmax benchmark
        {"name": "softmax 16384x4096", "family": "softmax", "n": 16384, "m": 4096, "dtype": "f32", "threads": 512},
        # half precision, rows that are no whole number of vectors or of threads
        {"name": "softmax 5000x1777 half", "family": "softmax", "n": 5000, "m": 1777, "dtype": "f16", "threads": 256},
        # the SDDMM benchmark
        {"name": "sddmm 8192 k128", "family": "sddmm", "n": 8192, "k": 128, "per_row": 82, "dtype": "f32", "csr": False},
        # a sparse solver's inner product: double precision, rows of uneven length
        {"name": "spmv 100000 double", "family": "spmv", "n": 100000, "avg": 50, "dtype": "f64"},
        # aggregation over a graph's neighbours: 128 features
        {"name": "spmm 20000x128", "family": "spmm", "n": 20000, "avg": 24, "cols": 128, "dtype": "f32"},
        # a relaxation whose time loop stays on the host: two launches per step
        {"name": "jacobi 1000003", "family": "jacobi", "n": 1000003, "steps": 50, "dtype": "f64"},
        # the forward-pass benchmark's 5-mer configuration, the user code as it is ported
        {"name": "hmm 5-mer", "family": "hmm", "k": 5, "form": "reference", "reads": 100, "min_len": 5000, "max_len": 15000},
        # the headline: 7-mer configuration, scaled linear space
        {"name": "hmm 7-mer scaled", "family": "hmm", "k": 7, "form": "scaled", "reads": 100, "min_len": 5000, "max_len": 15000},
        # the largest: the 16-layer model of 7-mers (262144 states), unchanged user code, one launch per step
        {"name": "hmm16 7-mer", "family": "hmm16", "k": 7, "form": "reference", "reads": 100, "min_len": 500, "max_len": 1500},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case; element counts and step counts keep it below the largest listed one."""
    family = rng.choice(("rows", "rows", "softmax", "softmax", "sddmm", "spmv", "spmm", "jacobi", "hmm", "hmm16"))
    if family == "rows":
        n = _log_int(rng, 1, 16384)
        m = _log_int(rng, 100, min(10000000, 100000000 // n))
        dtype = rng.choice(("f32", "f32", "f64"))
        threads = rng.choice((64, 128, 256, 512, 1024)) if m < 200000 or n > 64 else rng.choice((8192, 32768))
        return {"family": family, "n": n, "m": m, "dtype": dtype, "threads": threads}
    if family == "softmax":
        m = _log_int(rng, 64, 32768)
        n = _log_int(rng, 16, max(17, min(65536, 67108864 // m)))
        return {"family": family, "n": n, "m": m, "dtype": rng.choice(("f32", "f32", "f16", "f64")),
                "threads": rng.choice((128, 256, 512) if m < 4096 else (256, 512, 1024))}
    if family == "sddmm":
        n = _log_int(rng, 500, 16384)
        k = rng.choice((64, 128, 1024, _log_int(rng, 32, 1024)))
        per_row = max(1, min(n // 2, _log_int(rng, 2, max(3, min(200, 400000000 // (n * k))))))
        return {"family": family, "n": n, "k": k, "per_row": per_row, "dtype": rng.choice(("f32", "f32", "f64")), "csr": rng.random() < 0.5}
    if family == "spmv":
        n = _log_int(rng, 1000, 1000000)
        return {"family": family, "n": n, "avg": _log_int(rng, 4, max(5, min(200, 10000000 // n))), "dtype": rng.choice(("f32", "f64"))}
    if family == "spmm":
        n = _log_int(rng, 1000, 100000)
        cols = rng.choice((32, 64, 128, 256, rng.randint(33, 256)))
        return {"family": family, "n": n, "avg": _log_int(rng, 4, max(5, min(64, 100000000 // (n * cols)))), "cols": cols, "dtype": "f32"}
    if family == "jacobi":
        return {"family": family, "n": _log_int(rng, 1000, 4000000), "steps": _log_int(rng, 5, 100), "dtype": rng.choice(("f32", "f64"))}
    max_len = _log_int(rng, 200, 15000)
    if family == "hmm":
        k = rng.choice((3, 4, 5, 6, 7))
        form = rng.choice(("reference", "grouped", "scaled"))
        if k == 7 and form != "scaled":
            max_len = min(max_len, 8000)
        return {"family": family, "k": k, "form": form, "reads": rng.randint(20, 200), "min_len": max_len // 3, "max_len": max_len}
    k = rng.choice((3, 4, 5, 6, 7))
    form = "reference" if k > 5 else rng.choice(("reference", "scaled"))
    max_len = min(max_len, {3: 8000, 4: 8000, 5: 8000, 6: 2000, 7: 1500}[k])
    return {"family": family, "k": k, "form": form, "reads": rng.randint(20, 100), "min_len": max_len // 3, "max_len": max_len}


# ---------------------------------------------------------------- inputs
class _Source:
    """Seeded random tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def uniform(self, shape, lo, hi, dtype=torch.float32):
        x = torch.rand(shape, generator=self.g, device="cuda", dtype=torch.float32 if dtype == torch.float16 else dtype)
        return (x * (hi - lo) + lo).to(dtype)

    def normal(self, shape, dtype=torch.float32):
        return torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32 if dtype == torch.float16 else dtype).to(dtype)

    def integers(self, shape, lo, hi, dtype=torch.int64):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=dtype)

    def log_dirichlet(self, rows, parts):
        """Logarithms of `rows` draws from a flat Dirichlet distribution over `parts` probabilities, [rows, parts]."""
        e = -torch.log1p(-torch.rand((rows, parts), generator=self.g, device="cuda", dtype=torch.float64)).clamp_min(1e-12)
        return torch.log(e / e.sum(1, keepdim=True)).to(torch.float32)


def _uneven_csr(src, n, m, avg, dtype):
    """n x m matrix of n * avg non-zeros whose rows differ in length (a tenth of the rows hold about a third of them)."""
    nnz = n * avg
    u = torch.rand(nnz, generator=src.g, device="cuda", dtype=torch.float64)
    row = (u.pow(2.0) * n).to(torch.int64).clamp_max(n - 1)
    order = torch.randperm(n, generator=src.g, device="cuda")
    counts = torch.bincount(order[row], minlength=n)
    crows = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    crows[1:] = torch.cumsum(counts, 0)
    return {"values": src.normal(nnz, dtype), "rows": crows, "cols": src.integers((nnz,), 0, m), "nrows": n}


def _mask(src, n, per_row, dtype):
    """n x n mask with `per_row` distinct ascending columns in every row."""
    cols = src.integers((n, per_row), 0, n - per_row + 1).sort(1).values + torch.arange(per_row, device="cuda")
    rows = torch.arange(n, device="cuda").repeat_interleave(per_row)
    crows = torch.arange(n + 1, device="cuda") * per_row
    return crows, rows, cols.reshape(-1).contiguous(), src.normal(n * per_row, dtype)


def _reads(src, reads, min_len, max_len):
    """A padded batch of observation sequences; the longest read has the padded length."""
    lens = src.integers((reads,), min_len, max_len + 1)
    lens[int(reads // 2)] = max_len
    data = src.integers((reads, max_len), 0, OBSERVATIONS, torch.int8)
    data[torch.arange(max_len, device="cuda")[None, :] >= lens[:, None]] = 0
    return {"data": data, "lens": lens, "maxlen": max_len, "num_instances": reads}


def _synthetic_model(src, k):
    states = 4 ** k
    p = src.log_dirichlet(states, 5)
    return {"trans1": p[:, :4].contiguous(), "stay": p[:, 4].contiguous(), "output_prob": src.log_dirichlet(states, OBSERVATIONS).T.contiguous(),
            "initial_prob": torch.full((states,), -math.log(states), device="cuda"), "num_states": states}


def _layered_model(src, k, tail=0.05):
    kmers = 4 ** k
    init = torch.full((16 * kmers,), -math.inf, device="cuda")
    init[:kmers] = -math.log(kmers)
    return {"trans1": src.log_dirichlet(kmers, 4), "trans2": src.log_dirichlet(1, 16)[0].contiguous(),
            "output_prob": src.log_dirichlet(kmers, OBSERVATIONS).T.contiguous(), "initial_prob": init,
            "gamma": torch.tensor(math.log(tail), device="cuda"), "synthetic_248": torch.tensor(math.log1p(-tail), device="cuda"),
            "num_states": 16 * kmers}


def _work_of_a_step(case):
    """Operations per state and step (an exponential or a logarithm counts as one)."""
    return {"scaled": 11, "grouped": 17, "reference": 27}[case["form"]]


def _states(case):
    return 4 ** case["k"] * (16 if case["family"] == "hmm16" else 1)


def prepare(case, seed):
    src = _Source(seed)
    family = case["family"]
    s = {"case": dict(case)}
    if family in ("hmm", "hmm16"):
        states, reads = _states(case), case["reads"]
        layered = family == "hmm16"
        model = _layered_model(src, case["k"]) if layered else _synthetic_model(src, case["k"])
        if case["form"] != "reference":
            model = W.scaled_tables_on_device(model, reference_format=layered)
        s["model"], s["seqs"] = model, _reads(src, reads, case["min_len"], case["max_len"])
        s["a1"] = torch.zeros((reads, states), device="cuda")
        s["a2"] = torch.zeros((reads, states), device="cuda")
        s["result"] = torch.zeros(reads, dtype=torch.float64 if case["form"] == "scaled" else torch.float32, device="cuda")
        return s
    dtype = DTYPES[case["dtype"]]
    n = case["n"]
    if family == "rows":
        s["x"], s["out"] = src.uniform((n, case["m"]), -1.0, 1.0, dtype), torch.zeros(n, dtype=dtype, device="cuda")
    elif family == "softmax":
        s["x"] = src.normal((n, case["m"]), dtype)
        s["out"] = torch.zeros_like(s["x"])
    elif family == "sddmm":
        crows, rows, cols, values = _mask(src, n, case["per_row"], dtype)
        s["A"], s["B"] = src.normal((n, case["k"]), dtype), src.normal((case["k"], n), dtype)
        s["C"] = {"cols": cols, "values": values, "nnz": n * case["per_row"]}
        if case["csr"]:
            s["C"].update(crows=crows, rows=torch.zeros_like(rows))
        else:
            s["C"]["rows"] = rows
        s["D"] = torch.zeros_like(values)
    elif family == "spmv":
        s["A"], s["x"], s["y"] = _uneven_csr(src, n, n, case["avg"], dtype), src.normal(n, dtype), torch.zeros(n, dtype=dtype, device="cuda")
    elif family == "spmm":
        s["A"] = _uneven_csr(src, n, n, case["avg"], dtype)
        s["B"] = {"values": src.normal((n, case["cols"]), dtype), "ncols": case["cols"]}
        s["C"] = torch.zeros((n, case["cols"]), dtype=dtype, device="cuda")
    else:
        s["A"], s["B"] = src.normal(n, dtype), src.normal(n, dtype)
    return s


# ---------------------------------------------------------------- the call
def run(state):
    case = state["case"]
    family = case["family"]
    if family == "rows":
        W.sum_rows(state["x"], state["out"], case["n"],
                   opts=parpy.par({'outer': parpy.threads(case["n"]), 'inner': parpy.threads(case["threads"])}))
        return state["out"]
    if family == "softmax":
        W.softmax(state["x"], case["n"], case["m"], state["out"],
                  opts=parpy.par({'N': parpy.threads(case["n"]), 'M': parpy.threads(case["threads"])}))
        return state["out"]
    if family == "sddmm":
        nnz = state["C"]["nnz"]
        if case["csr"]:
            W.sddmm_csr(state["A"], state["B"], state["C"], state["D"], case["n"], 1.0, 0.5,
                        opts=parpy.par({'N': parpy.threads(case["n"]), 'M': parpy.threads(64), 'nnz': parpy.threads(nnz).tpb(256)}))
            return state["D"], state["C"]["rows"]
        W.sddmm_coo(state["A"], state["B"], state["C"], state["D"], 1.0, 0.5, opts=parpy.par({'nnz': parpy.threads(nnz).tpb(256)}))
        return state["D"]
    if family == "spmv":
        spmv(state["A"], state["x"], state["y"], opts=parpy.par({'row': parpy.threads(case["n"])}))
        return state["y"]
    if family == "spmm":
        spmm(state["A"], state["B"], state["C"], opts=parpy.par({'i': parpy.threads(case["n"]), 'j': parpy.threads(case["cols"])}))
        return state["C"]
    if family == "jacobi":
        jacobi(case["steps"], state["A"], state["B"], opts=parpy.par({'N': parpy.threads(case["n"]).tpb(256)}))
        return state["A"], state["B"]
    model, seqs, a1, a2, result = (state[k] for k in ("model", "seqs", "a1", "a2", "result"))
    states, form = _states(case), case["form"]
    if family == "hmm":
        f = {"reference": W.forward_syn, "grouped": W.forward_syn4, "scaled": W.forward_scaled}[form]
        threads = parpy.threads(min(1024, states if form == "reference" else states // 4))
        f(model, seqs, result, a1, a2, opts=parpy.par({'inst': parpy.threads(case["reads"]), 'state': threads}))
    elif form == "scaled":
        opts = parpy.par({'inst': parpy.threads(case["reads"]), 'state': parpy.threads(min(1024, states // 16))})
        W.forward_kernel_scaled(model, seqs, result, a1, a2, opts=opts)
    else:
        # a model that fits a workgroup runs whole in one; a larger one has a thread per k-mer and the time loop on the host
        threads = parpy.threads(min(1024, states)) if states <= 16384 else parpy.threads(states // 16).tpb(256)
        W.forward_kernel(model, seqs, a1, a2, result, opts=parpy.par({'inst': parpy.threads(case["reads"]), 'state': threads}))
    return result, a1, a2


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    family = case["family"]
    if family in ("hmm", "hmm16"):
        states, kmers, reads = _states(case), 4 ** case["k"], case["reads"]
        steps = reads * (case["min_len"] + case["max_len"]) / 2
        return {"bytes": 4 * kmers * (OBSERVATIONS + 5) + 4 * states + steps + 8 * reads * states, "flops": steps * states * _work_of_a_step(case)}
    size, n = SIZEOF[case["dtype"]], case["n"]
    if family == "rows":
        return {"bytes": size * (n * case["m"] + n), "flops": n * case["m"]}
    if family == "softmax":
        return {"bytes": 2 * size * n * case["m"], "flops": 5 * n * case["m"]}
    if family == "sddmm":
        nnz = n * case["per_row"]
        index = 8 * nnz + (8 * (n + 1 + nnz) if case["csr"] else 8 * nnz)
        return {"bytes": size * (2 * n * case["k"] + 2 * nnz) + index, "flops": nnz * (2 * case["k"] + 3)}
    if family == "spmv":
        nnz = n * case["avg"]
        return {"bytes": (size + 8) * nnz + 8 * (n + 1) + 2 * size * n, "flops": 2 * nnz}
    if family == "spmm":
        nnz = n * case["avg"]
        return {"bytes": (size + 8) * nnz + 8 * (n + 1) + 2 * size * n * case["cols"], "flops": 2 * nnz * case["cols"]}
    return {"bytes": 3 * size * n, "flops": 8 * (case["steps"] - 1) * n}


def tolerance(case):
    family = case["family"]
    if family in ("hmm", "hmm16"):
        # log space: rounding of scores of up to 1e5 over the steps; linear space: relative rounding of 15000 products
        return {"rel": 1e-4} if case["form"] == "scaled" else {"rel": 1e-5}
    return {"rel": {"f16": 5e-3, "f32": 1e-5, "f64": 1e-12}[case["dtype"]]}
