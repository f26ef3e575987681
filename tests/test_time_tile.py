"""Time loops over element-wise updates from shifted elements: several steps per launch against one launch per update
(`opt_tile_steps` off), at array lengths around the stretches of a wavefront."""
import numpy as np
import pytest

import parpy_amd as parpy
from parpy_amd.compile import hiprtc_compile
from parpy_amd.operators import float32, max

HIP = parpy.CompileBackend.Hip


def jacobi(A, B, C, n, steps):
    for t in range(1, steps):
        parpy.label('N')
        B[1:-1] = (A[:-2] + A[1:-1] + A[2:]) / 3.0
        parpy.label('N')
        A[1:-1] = (B[:-2] + B[1:-1] + B[2:]) / 3.0


def wave_equation(A, B, C, n, steps):
    """One update per step, reach two, a coefficient array, the own element of the array it writes."""
    for t in range(steps):
        parpy.label('N')
        for i in range(2, n - 3):
            s = A[i - 2] + A[i + 2] - A[i] * 2.0
            B[i] = A[i] * 1.5 - B[i] * 0.5 + C[i] * s / 7.0
        parpy.label('N')
        for i in range(1, n):
            A[i] = max(B[i - 1], A[i] * 0.25) + 0.001 * B[i]


def lopsided(A, B, C, n, steps):
    """Two arrays written by one launch, one-sided reach, the iteration number as a value."""
    for t in range(steps):
        parpy.label('N')
        for i in range(n - 1):
            A[i] = C[i + 1] * 0.5 + A[i] * 0.5
            B[i] = A[i] + float32(i % 5)
        parpy.label('N')
        for i in range(3, n):
            C[i] = B[i - 3] * 0.125 + C[i] * 0.875


def driven(A, B, C, n, steps):
    """An array that the loop only reads, which a caller may pass a second time under the name of one it writes."""
    for t in range(steps):
        parpy.label('N')
        B[1:-1] = (A[:-2] + A[2:]) * 0.5
        parpy.label('N')
        A[1:-1] = B[1:-1] * 0.25 + C[2:]


PROGRAMS = [jacobi, wave_equation, lopsided]


def run(f, arrays, n, steps, **kw):
    o = parpy.par({'N': parpy.threads(n)})
    o.backend = HIP
    for k, v in kw.items():
        setattr(o, k, v)
    got = [a.copy() for a in arrays]
    parpy.jit(f)(*got, n, steps, opts=o)
    return got


@pytest.mark.parametrize("f", PROGRAMS, ids=lambda f: f.__name__)
def test_steps_of_a_stencil_share_a_launch(f):
    o = parpy.par({'N': parpy.threads(5000)})
    o.backend = HIP
    args = [np.zeros(5000), np.zeros(5000), np.zeros(5000), 5000, 20]
    s = parpy.print_compiled(f, args, o)
    hiprtc_compile(s[:s.index("// host side")], o)
    assert "parpy_lane_before" in s and s[s.index("// host side"):].count("<<<") == 2
    o.opt_tile_steps = False
    s = parpy.print_compiled(f, args, o)
    assert "parpy_lane_before(" not in s[s.index('extern "C"'):]


@pytest.mark.gpu
@pytest.mark.parametrize("f", PROGRAMS, ids=lambda f: f.__name__)
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=lambda d: np.dtype(d).name)
def test_tiled_steps_match_one_launch_per_update(f, dtype):
    rng = np.random.default_rng(7)
    for n, steps in [(512, 3), (513, 50), (1000, 2), (1024, 17), (4093, 64), (20000, 7), (65537, 33), (800001, 12)]:
        arrays = [rng.standard_normal(n).astype(dtype) for _ in range(3)]
        arrays[0][n // 2] = 0.0
        arrays[0][n // 3] = 1e-42 if dtype == np.float32 else 5e-324
        want, got = run(f, arrays, n, steps, opt_tile_steps=False), run(f, arrays, n, steps)
        for w, g in zip(want, got):
            # (products and sums may be contracted to fused multiply-adds differently)
            same = np.array_equal(w, g) if f is jacobi else np.allclose(w, g, rtol=1e-12 if dtype == np.float64 else 1e-4, atol=1e-13 if dtype == np.float64 else 1e-5)
            assert same, (f.__name__, n, steps, np.abs(w - g).max())


def plan_of(f, args, o):
    o = parpy.backend._resolve_backend(o, False)
    return parpy.compiler.compile_ir(parpy._ir_asts[parpy.jit(f)], parpy.validate.check_arguments(args, o, False), o, {}).plan


def test_a_written_array_must_not_be_reachable_under_another_name():
    """The plan tests every pair of arrays of which one is written, over their whole length, and keeps the loop of launches."""
    import re
    o = parpy.par({'N': parpy.threads(5000)})
    o.backend = HIP
    plan = plan_of(driven, [np.zeros(5000, dtype=np.float32) for _ in range(3)] + [5000, 20], o)
    pairs = re.findall(r'\(disjoint \(v "?(\w)_\d+"?\) \(i 20000\) \(v "?(\w)_\d+"?\) \(i 20000\)\)', plan)
    assert sorted("".join(sorted(p)) for p in pairs) == ["AB", "AC", "BC"]
    tiled, updates = re.search(r"\(then (.*)\) \(else (.*)\)\)", plan).groups()
    assert tiled.count("(launch") == 2 and updates.count("(launch") == 2 and "(i 20)" in updates


def decay(A, n, steps):
    for t in range(steps):
        parpy.label('N')
        for i in range(n):
            A[i] = A[i] * 0.5 + 1.0
        parpy.label('N')
        A[1:] = A[1:] - 0.25


def test_a_call_does_not_need_memory_for_the_second_set_of_arrays():
    """Whatever its size, the plan holds the loop of launches for a run that cannot have it."""
    import re
    o = parpy.par({'N': parpy.threads(5000)})
    o.backend = HIP
    for f, args in ((decay, [np.zeros(5000)]), (driven, [np.zeros(5000) for _ in range(3)]), (jacobi, [np.zeros(3000000) for _ in range(3)])):
        plan = plan_of(f, args + [len(args[0]), 20], o)
        assert re.search(r"\(if .*\(fits \d+\)\)? \(then \(alloc .*\(launch .*\) \(else \(for .*\(launch ", plan)


def test_few_updates_of_long_arrays_stay_launches():
    o = parpy.par({'N': parpy.threads(5000)})
    o.backend = HIP
    for n, dtype, steps, tiled in ((5000, np.float64, 3, True), (799999, np.float64, 3, True), (800000, np.float64, 3, False),
                                   (800000, np.float64, 4, True), (800000, np.float32, 3, True), (5000, np.float64, 2, False)):
        a = np.empty(n, dtype=dtype)
        assert ("parpy_lane_before(" in parpy.print_compiled(jacobi, [a, a, a, n, steps], o).split('extern "C"', 1)[1]) == tiled, (n, dtype, steps)


def test_second_sets_that_no_pool_hands_out_quickly_are_not_asked_for():
    o = parpy.par({'N': parpy.threads(5000)})
    o.backend = HIP
    for n, tiled in ((400_000_000, True), (600_000_000, False)):   # two float64 arrays: 6.4 and 9.6 GB
        a = np.empty(n)   # (never touched)
        assert ("parpy_lane_before(" in parpy.print_compiled(jacobi, [a, a, a, n, 10], o).split('extern "C"', 1)[1]) == tiled


@pytest.mark.gpu
def test_a_branch_whose_temporaries_are_refused_is_not_taken():
    """Through the runtime's own entry points: the first temporary can be had, the second (4 TiB) cannot."""
    import ctypes
    torch = pytest.importorskip("torch")
    from parpy_amd import runtime
    o = parpy.par({})
    o.backend = HIP
    lib = runtime._compile_runtime_lib(HIP)
    code = hiprtc_compile('extern "C" __global__ void add(float* x, float v) { if (threadIdx.x == 0) x[0] += v; }', o)
    buf, module = ctypes.create_string_buffer(code, len(code)), ctypes.c_void_p()
    assert lib.parpy_hip_module_load(buf, len(code), ctypes.byref(module)) == 0
    x = torch.zeros(1, device="cuda")
    arr = (ctypes.c_void_p * 1)(x.data_ptr())

    def plan(second):
        text = ('(plan "f" (params ("x" ptr)) (kernels ("add" (params ptr f32))) (body (if (bin and i (i 1) (fits 1)) (then (alloc "t" 1024) '
                f'(alloc "u" {second}) (launch 0 1 1 1 64 1 1 (args (v "t") (f 1))) (launch 0 1 1 1 64 1 1 (args (v "x") (f 1))) (free "t") (free "u") ) '
                '(else (launch 0 1 1 1 64 1 1 (args (v "x") (f 100))) )) (launch 0 1 1 1 64 1 1 (args (v "x") (f 1000))) ))')
        h = ctypes.c_void_p()
        assert lib.parpy_hip_plan_create(module, text.encode(), ctypes.byref(h)) == 0, lib.parpy_get_error_message()
        return h

    total = 0.0
    for second, run, adds in ((4096, lib.parpy_hip_plan_run, 1001.0), (1 << 42, lib.parpy_hip_plan_run, 1100.0),
                              (4096, lib.parpy_hip_plan_run_noalloc, 1001.0), (1 << 24, lib.parpy_hip_plan_run_noalloc, 1100.0)):
        h = plan(second)
        for graph in (0, 1) if run is lib.parpy_hip_plan_run else (0,):
            lib.parpy_hip_plan_set_graph(h, graph)
            for _ in range(4):
                assert run(h, arr, 1) == 0, lib.parpy_get_error_message()
                total += adds
                assert lib.parpy_sync() == 0 and x.item() == total, (second, graph)
            assert lib.parpy_hip_plan_launch_count(h) == (3 if adds == 1001.0 else 2)
        assert lib.parpy_hip_plan_destroy(h) == 0


@pytest.mark.gpu
def test_arrays_passed_under_two_names():
    torch = pytest.importorskip("torch")
    n, steps = 4000, 12
    f = parpy.jit(driven)

    def call(arrays, **kw):
        o = parpy.par({'N': parpy.threads(n)})
        for k, v in kw.items():
            setattr(o, k, v)
        f(*arrays, n, steps, opts=o)
        parpy.sync(HIP)
        o = parpy.backend._resolve_backend(o, True)
        return parpy._compile_function(parpy._ir_asts[f], parpy.validate.check_arguments([*arrays, n, steps], o, True), o).launch_count()

    def arrays(overlap, seed):
        """A and B apart; C is B (None) or starts `overlap` elements before B ends."""
        g = torch.Generator(device="cuda").manual_seed(seed)
        buf = torch.randn(3 * n, generator=g, device="cuda")
        A, B = buf[:n], buf[n:2 * n]
        return buf, [A, B, B if overlap is None else buf[2 * n - overlap:3 * n - overlap]]

    for q, (overlap, tiled) in enumerate([(None, False), (0, True), (4, False), (n, False)]):
        whole, a = arrays(overlap, q)
        want, b = arrays(overlap, q)
        assert call(a) == (2 if tiled else 2 * steps), overlap
        call(b, opt_tile_steps=False)
        # (products and sums may be contracted to fused multiply-adds differently)
        assert torch.allclose(whole, want, rtol=1e-4, atol=1e-5), overlap
