"""Time loops on the host over two arrays that change places: two steps per launch against one launch per step
(`opt_tile_steps` off), rows that end at every place of a launch, numbers of steps around the pairs of launches."""
import re

import numpy as np
import pytest

import parpy_amd as parpy
from parpy_amd import workloads as W
from parpy_amd.compile import hiprtc_compile
from parpy_amd.operators import exp, int32, int8, log, max

HIP = parpy.CompileBackend.Hip
R, S, N = 5, 1024, 128      # rows, elements, threads of a row: eight elements a thread


@parpy.jit
def quads(x, a, b, p, q, lens, n, steps):
    """What four neighbours share: evenly apart, and the thread's next element; rows end."""
    parpy.label('r')
    for r in range(n):
        for t in range(1, steps):
            src = b
            dst = a
            if t & 1:
                src = a
                dst = b
            o = x[r, t]
            parpy.label('s')
            for s in range(1024):
                if t < lens[r]:
                    u = int32((s // 4) % 32)
                    v = max(src[r, u] * p[s % 4], src[r, 32 + u]) + src[r, 64 + u] - src[r, 96 + u] * p[s // 128]
                    w = 1 if s // 128 == 7 else s // 128 + 1
                    if s // 128 == 7:
                        w = 7
                    v = v * 0.25 + src[r, w * 128 + s % 128] * 0.5
                    dst[r, s] = v + q[o, s % 128]
                elif t == lens[r]:
                    dst[r, s] = src[r, s]


@parpy.jit
def one_other(x, a, b, p, q, lens, n, steps):
    """A single element of another thread, one that no four threads have in common; rows that do not end."""
    parpy.label('r')
    for r in range(n):
        for t in range(2, steps):
            src = b
            dst = a
            if t & 1:
                src = a
                dst = b
            parpy.label('s')
            for s in range(1024):
                dst[r, s] = src[r, s] * 0.5 + src[r, 256 + (s % 128 + 3) % 128] * p[s // 128] + q[x[r, t], s % 128]


@parpy.jit
def product_last(x, a, b, p, q, lens, n, steps):
    """An update that ends in a product, which the next step adds to another: rounded in between."""
    parpy.label('r')
    for r in range(n):
        for t in range(1, steps):
            src = b
            dst = a
            if t & 1:
                src = a
                dst = b
            parpy.label('s')
            for s in range(1024):
                if t < lens[r]:
                    dst[r, s] = (src[r, s] + src[r, (s // 4) % 32]) * p[s // 128]
                elif t == lens[r]:
                    dst[r, s] = src[r, s]


@parpy.jit
def four_others(x, a, b, p, q, lens, n, steps):
    """Four elements of others, not evenly apart: half of a thread's own, too many to compute again."""
    parpy.label('r')
    for r in range(n):
        for t in range(1, steps):
            src = b
            dst = a
            if t & 1:
                src = a
                dst = b
            parpy.label('s')
            for s in range(1024):
                u = (s // 4) % 32
                dst[r, s] = (src[r, u] + src[r, 33 + u] + src[r, 64 + u] + src[r, 96 + u]) * 0.125 + src[r, s] * p[s // 128]


@parpy.jit
def looked_up(x, a, b, p, q, lens, n, steps):
    """Elements whose place stands in memory."""
    parpy.label('r')
    for r in range(n):
        for t in range(1, steps):
            src = b
            dst = a
            if t & 1:
                src = a
                dst = b
            parpy.label('s')
            for s in range(1024):
                dst[r, s] = src[r, x[r, s % 16]] * 0.5 + src[r, s] * p[s // 128]


@parpy.jit
def cut_short(x, a, b, p, q, lens, n, steps):
    """A place that passes through eight bits: not the number that it is made of."""
    parpy.label('r')
    for r in range(n):
        for t in range(1, steps):
            src = b
            dst = a
            if t & 1:
                src = a
                dst = b
            parpy.label('s')
            for s in range(1024):
                u = 128 + int8(s % 128 + 100)
                dst[r, s] = src[r, u] * 0.5 + src[r, s] * p[s // 128]


@parpy.jit
def goes_on(x, a, b, p, q, lens, n, steps):
    """Rows that stop without a copy: the arrays end two steps apart."""
    parpy.label('r')
    for r in range(n):
        for t in range(1, steps):
            src = b
            dst = a
            if t & 1:
                src = a
                dst = b
            parpy.label('s')
            for s in range(1024):
                if t < lens[r]:
                    dst[r, s] = src[r, (s // 4) % 32] * 0.25 + src[r, s] * p[s // 128]


def options(**kw):
    o = parpy.par({'r': parpy.threads(R), 's': parpy.threads(N).tpb(64)})
    o.backend = HIP
    for k, v in kw.items():
        setattr(o, k, v)
    return o


def arguments(steps, lens, dtype, seed=1):
    rng = np.random.default_rng(seed)
    return [rng.integers(0, 6, (R, max(steps, 16))).astype(np.int8), rng.standard_normal((R, S)).astype(dtype), rng.standard_normal((R, S)).astype(dtype),
            rng.standard_normal(8).astype(dtype), rng.standard_normal((6, 128)).astype(dtype), np.array(lens, np.int64), R, steps]


@pytest.mark.parametrize("fn,joined", [(quads, True), (one_other, True), (product_last, True), (four_others, False), (looked_up, False), (cut_short, False), (goes_on, False)])
def test_which_loops(fn, joined):
    s = parpy.print_compiled(fn, arguments(40, [40] * R, np.float32), options())
    hiprtc_compile(s[:s.index("// host side")], options())
    assert ("_two_steps_" in s) == joined
    assert ("parpy_dpp<85>(" in s.split('extern "C"', 1)[1]) == (fn is quads)
    for steps in (1, 8, 9):      # eight steps behind the first two make two pairs of launches
        s = parpy.print_compiled(fn, arguments(steps, [steps] * R, np.float32), options())
        assert "_two_steps_" not in s
    assert "_two_steps_" not in parpy.print_compiled(fn, arguments(40, [40] * R, np.float32), options(opt_tile_steps=False))


@pytest.mark.parametrize("fn,product", [(quads, False), (product_last, True)])
def test_products_between_are_rounded(fn, product):
    s = parpy.print_compiled(fn, arguments(40, [40] * R, np.float32), options())
    between = re.findall(r"float between_\d+ = (.*);", s)
    assert len(between) > 8
    for value in between:
        assert value.startswith("parpy_dpp<") or value.startswith("parpy_rounded(") == product


def test_arrays_that_overlap_run_as_single_steps():
    """The plan compares the two arrays with each other and with all others and holds the loop of single steps beside the rest."""
    args, o = arguments(40, [40] * R, np.float32), parpy.backend._resolve_backend(options(), False)
    plan = parpy.compiler.compile_ir(parpy._ir_asts[quads], parpy.validate.check_arguments(args, o, False), o, {}).plan
    pairs = {frozenset(m) for m in re.findall(r'\(disjoint \(v "?(\w+?)_\d+"?\) \(i \d+\) \(v "?(\w+?)_\d+"?\) \(i \d+\)\)', plan)}
    assert pairs == {frozenset(q) for q in ("ab", "ax", "ap", "aq", ("a", "lens"), "bx", "bp", "bq", ("b", "lens"))}
    joined, single = re.search(r"\(then (.*)\) \(else (.*)\)\)", plan).groups()
    assert joined.count("(launch") == 4 and single.count("(launch") == 1 and "(i 40)" in single


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("steps", [10, 11, 12, 13, 14, 31])
def test_rows_end_everywhere(steps, dtype):
    ends = list(range(0, steps + 3)) + [-1, 100]
    ends += [steps] * (-len(ends) % R)
    for q in range(0, len(ends), R):
        got, want = arguments(steps, ends[q:q + R], dtype), arguments(steps, ends[q:q + R], dtype)
        for fn in (quads, product_last):
            fn(*got, opts=options())
            fn(*want, opts=options(opt_tile_steps=False))
            assert np.array_equal(got[1], want[1]) and np.array_equal(got[2], want[2]), (steps, ends[q:q + R])


@pytest.mark.gpu
@pytest.mark.parametrize("fn", [one_other, four_others, looked_up, cut_short, goes_on])
def test_other_loops(fn):
    for steps in (11, 12, 18, 41):
        got, want = arguments(steps, [3, 9, 10, steps - 1, steps], np.float32), arguments(steps, [3, 9, 10, steps - 1, steps], np.float32)
        fn(*got, opts=options())
        fn(*want, opts=options(opt_tile_steps=False))
        assert np.array_equal(got[1], want[1]) and np.array_equal(got[2], want[2]), (fn, steps)


@pytest.mark.gpu
def test_a_table_inside_one_of_the_arrays():
    """`p` is the first elements of a row that no step writes any more: a launch for two steps would not see what is stored there."""
    import torch
    results = []
    for tiled in (True, False):
        x, a, b, p, q, lens, n, steps = [torch.from_numpy(v).cuda() if isinstance(v, np.ndarray) else v for v in arguments(20, [20, 20, 20, 20, 0], np.float32)]
        quads(x, a, b, a[4, 8:16], q, lens, n, steps, opts=options(opt_tile_steps=tiled))
        parpy.sync(HIP)
        o = parpy.backend._resolve_backend(options(opt_tile_steps=tiled), True)
        call = [x, a, b, a[4, 8:16], q, lens, n, steps]
        launches = parpy._compile_function(parpy._ir_asts[quads], parpy.validate.check_arguments(call, o, True), o).launch_count()
        assert launches == 19, tiled
        results.append((a, b))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])


@pytest.mark.gpu
@pytest.mark.parametrize("graphs", [False, True])
def test_layers(graphs):
    """The 16-layer model with a thread per state of a layer, also replayed from a graph; the same arrays on every call."""
    import torch
    k, reads, steps = 4, 6, 45
    rng = np.random.default_rng(3)
    kmers = 4 ** k
    hmm = W.to_device({"trans1": np.log(rng.dirichlet(np.ones(4), kmers)).astype(np.float32), "trans2": np.log(rng.dirichlet(np.ones(16))).astype(np.float32),
                       "output_prob": np.ascontiguousarray(np.log(rng.dirichlet(np.ones(101), kmers)).T.astype(np.float32)),
                       "initial_prob": np.concatenate([np.full(kmers, -np.log(kmers)), np.full(15 * kmers, -np.inf)]).astype(np.float32),
                       "gamma": np.float32(np.log(0.05)), "synthetic_248": np.float32(np.log1p(-0.05)), "num_states": 16 * kmers})
    seqs = W.to_device({"data": rng.integers(0, 101, (reads, steps)).astype(np.int8), "lens": np.array([steps, 44, 43, 30, 9, 2], np.int64),
                        "maxlen": steps, "num_instances": reads})
    kept = {}
    for tiled in (False, True):
        a1, a2 = (torch.zeros((reads, 16 * kmers), device="cuda") for _ in range(2))
        result = torch.zeros(reads, device="cuda")
        o = parpy.par({'inst': parpy.threads(reads), 'state': parpy.threads(kmers).tpb(64)})
        o.backend, o.opt_tile_steps, o.use_cuda_graphs = HIP, tiled, graphs
        for _ in range(4 if graphs else 1):
            a1.fill_(1.0), a2.fill_(2.0)
            W.forward_kernel(hmm, seqs, a1, a2, result, opts=o)
            parpy.sync(HIP)
            now = [x.clone() for x in (a1, a2, result)]
            if tiled:
                assert all(torch.equal(x, y) for x, y in zip(now, kept["single"]))
            else:
                kept["single"] = now
