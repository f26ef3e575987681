"""The call extension: which calls it takes for the same, and that what it runs is what the Python path would run."""
import ctypes

import numpy as np
import pytest

import parpy_amd as parpy
from parpy_amd.options import CompileOptions, LoopPar

torch = pytest.importorskip("torch")
HIP = parpy.CompileBackend.Hip


def opts(n=64, **kw):
    o = parpy.par({'N': parpy.threads(n)})
    for k, v in kw.items():
        setattr(o, k, v)
    return o


def test_calls_that_differ_in_anything_are_different_calls():
    from parpy_amd import fastcall
    ran = []
    run = ctypes.CFUNCTYPE(ctypes.c_int32, ctypes.c_void_p, ctypes.POINTER(ctypes.c_void_p), ctypes.c_int32)(lambda plan, p, n: ran.append(plan) or 0)
    table = fastcall._load().CallTable(CompileOptions, LoopPar, ctypes.cast(run, ctypes.c_void_p).value)
    f32 = lambda v: torch.tensor(v, dtype=torch.float32)
    calls = [((1,), opts()), ((1.0,), opts()), ((True,), opts()), ((2,), opts()), ((1, 1), opts()), (({"a": 1},), opts()), (({"b": 1},), opts()),
             (({"a": 1, "b": 2},), opts()), (({"a": 12},), opts()), ((f32(1.0),), opts()), ((f32(2.0),), opts()), ((torch.tensor(1.0, dtype=torch.float64),), opts()),
             ((1,), opts(128)), ((1,), opts(backend=HIP)), ((1,), opts(opt_vectorize=False)), ((1,), opts(opt_vectorize=True)), ((1,), opts(reg_budget=40)),
             ((1,), parpy.par({'M': parpy.threads(64)})), ((1,), parpy.par({'N': parpy.threads(64).reduce()})), ((1,), parpy.par({'N': parpy.threads(64).tpb(64)}))]
    for q, (args, o) in enumerate(calls):
        assert table.run(args, {"opts": o}) is None, q
        assert table.add(args, o, 1000 + q, ())
    for q, (args, o) in enumerate(calls):
        assert table.run(args, {"opts": o}) == 0 and ran[-1] == 1000 + q
    assert table.run((1,), {"opts": parpy.par({'N': parpy.threads(64)})}) == 0 and ran[-1] == 1000     # a fresh object with equal settings
    # what it leaves to the Python path
    for args, kw in [((1,), {}), ((1,), {"opts": opts(), "extra": 1}), ((1,), {"opts": None}), ((np.zeros(3),), {"opts": opts()}), ((torch.zeros(3),), {"opts": opts()}),
                     (({"a": {"b": 1}},), {"opts": opts()}), (({1: 1},), {"opts": opts()}), ((1 << 70,), {"opts": opts()}), ((1,), {"opts": opts(includes=["x"])})]:
        assert table.run(args, kw) is None
    table.clear()
    assert table.run((1,), {"opts": opts()}) is None


def test_tensors_without_memory_of_their_own_are_left_to_the_python_path():
    """Inside torch.vmap an argument is of type torch.Tensor and has no address; asking for it throws a C++ exception."""
    from parpy_amd import fastcall
    run = ctypes.CFUNCTYPE(ctypes.c_int32, ctypes.c_void_p, ctypes.POINTER(ctypes.c_void_p), ctypes.c_int32)(lambda plan, p, n: 0)
    table = fastcall._load().CallTable(CompileOptions, LoopPar, ctypes.cast(run, ctypes.c_void_p).value)
    answers = []

    def inside(v):
        for args in ((v,), ({"a": v, "b": 1},)):
            answers.append((type(v) is torch.Tensor, table.add(args, opts(), 1000, ()), table.run(args, {"opts": opts()})))
        return v
    torch.vmap(inside)(torch.zeros(3))                # 0-d
    torch.vmap(inside)(torch.zeros(3, 4))
    torch.func.grad(lambda v: inside(v) * 1.0)(torch.tensor(2.0))
    assert answers == [(True, False, None)] * 6
    assert table.add((torch.tensor(2.0),), opts(), 1000, ()) and table.run((torch.tensor(2.0),), {"opts": opts()}) == 0


def test_a_scalar_whose_memory_holds_its_negative_is_left_to_the_python_path():
    from parpy_amd import fastcall
    run = ctypes.CFUNCTYPE(ctypes.c_int32, ctypes.c_void_p, ctypes.POINTER(ctypes.c_void_p), ctypes.c_int32)(lambda plan, p, n: 0)
    table = fastcall._load().CallTable(CompileOptions, LoopPar, ctypes.cast(run, ctypes.c_void_p).value)
    v = torch.tensor(1 + 2j).conj().imag
    assert v.is_neg() and v.item() == -2.0
    assert not table.add((v,), opts(), 1000, ()) and table.run((torch.tensor(2.0),), {"opts": opts()}) is None
    assert table.run((v,), {"opts": opts()}) is None


def test_the_two_zeros_are_different_values():
    from parpy_amd.key import _describe_argument
    from parpy_amd.validate import check_arguments
    values = (0.0, -0.0, torch.tensor(0.0), torch.tensor(-0.0), 0, False, 1.5, 1, True)
    assert len({parpy._call_signature((x,))[0] for x in values}) == len(values)
    assert len({_describe_argument(check_arguments((x,), opts(backend=HIP), False)[0]) for x in values}) == len(values)


def plain_calls(monkeypatch, f):
    """`f` as a jitted function of scalars whose calls reach the warm path without a device; returns it and the list of its runs."""
    from parpy_amd import runtime
    ran = []

    def wrapper(*args):
        ran.append("checked")
    wrapper.run_pointers = lambda ptrs: ran.append("pointers")
    wrapper.lib, wrapper.plan = ctypes.CDLL(str(runtime.PARPY_HIP_BASE_LIB_PATH)), ctypes.c_void_p(1)
    monkeypatch.setattr(parpy, "_compile_function", lambda ir, args, opts: wrapper)
    monkeypatch.setattr(parpy.backend, "_resolve_backend", lambda opts, execute: opts)
    return parpy.jit(f), ran


def nothing(n):
    parpy.label('N')
    for i in range(n):
        t = i


def test_calls_run_without_the_extension(monkeypatch):
    """No compiler, no headers, a folder that cannot be written: said once, and not by a call that fails after its work is done."""
    import warnings
    from parpy_amd import fastcall
    tried = []

    def no_compiler(*a, **k):
        tried.append(1)
        raise RuntimeError("no compiler")
    monkeypatch.setattr(fastcall, "_module", None)
    monkeypatch.setattr(fastcall, "_unavailable", False, raising=False)
    monkeypatch.setattr(fastcall, "_command", no_compiler)
    f, ran = plain_calls(monkeypatch, nothing)
    with pytest.warns(RuntimeWarning, match="no compiler"):
        f(3, opts=opts())
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        f(3, opts=opts())
        f(4, opts=opts())
    assert ran == ["checked", "pointers", "checked"] and len(tried) == 1


def test_calls_that_the_extension_declines_are_offered_once(monkeypatch):
    from parpy_amd import fastcall
    offered = []
    order = fastcall.pointer_order
    monkeypatch.setattr(fastcall, "pointer_order", lambda args: offered.append(args) or order(args))
    f, ran = plain_calls(monkeypatch, nothing)
    for k in range(5):
        f(3, opts=opts(includes=["/usr/include"]))
    assert ran == ["checked"] + 4 * ["pointers"]
    assert len(offered) == 2      # under the state that was passed and the one after the backend was chosen
    for k in range(3):
        f(5, opts=opts(includes=["/usr/include"]))
    assert len(offered) == 4


def test_looking_for_the_extension_does_not_import_the_build_tools():
    import os
    import subprocess
    import sys
    code = "import sys, torch; from parpy_amd import fastcall; fastcall._load(); assert 'torch.utils.cpp_extension' not in sys.modules"
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    assert subprocess.run([sys.executable, "-W", "error::RuntimeWarning", "-c", code], cwd=root, timeout=300).returncode == 0


def test_plan_pointers_follow_the_sorted_fields():
    from parpy_amd import fastcall
    a, b, c, s = (torch.zeros(k) for k in (1, 2, 3, 4))
    assert fastcall.pointer_order((a, {"z": b, "n": 3, "c": c, "d": torch.tensor(1.0)}, 5, s)) == (0, 2, 1, 3)


def scale(d, out, n):
    parpy.label('N')
    for i in range(n):
        out[i] = d["x"][i] * d["w"] + d["b"][i]


@pytest.mark.gpu
def test_warm_calls_run_on_the_arguments_of_the_call():
    f = parpy.jit(scale)
    for rep in range(3):
        for n in (64, 65, 1000):
            for w in (2.0, 4.0):   # (exact products: a fused multiply-add rounds like the two operations)
                x, b = (torch.randn(n + 1, device="cuda") for _ in range(2))
                out = torch.full((n + 1,), -1.0, device="cuda")
                for off in (0, 1):                      # whole allocations and views that are only 4-byte aligned
                    xv, bv, ov = x[off:off + n], b[off:off + n], out[off:off + n]
                    fields = {"x": xv, "w": w, "b": bv} if rep % 2 else {"b": bv, "x": xv, "w": w}
                    f(fields, ov, n, opts=opts(256))
                    assert torch.equal(ov, xv * w + bv), (rep, n, w, off)
    z = torch.randn(64, device="cuda", requires_grad=True)
    with pytest.raises(Exception):
        f({"x": z, "w": 2.0, "b": z}, z, 64, opts=opts(256))
    parpy.clear_cache()
    out = torch.zeros(64, device="cuda")
    x = torch.randn(64, device="cuda")
    f({"x": x, "w": 2.0, "b": x}, out, 64, opts=opts(256))
    f({"x": x, "w": 2.0, "b": x}, out, 64, opts=opts(256))
    assert torch.equal(out, x * 2.0 + x)


@pytest.mark.gpu
def test_warm_calls_on_tensors_that_share_or_lack_memory():
    f = parpy.jit(scale)
    x, b = (torch.randn(64, device="cuda") for _ in range(2))
    out = torch.full((64,), -1.0, device="cuda")
    call = lambda o: f({"x": x, "w": 2.0, "b": b}, o, 64, opts=opts(64))
    call(out.clone())
    shared = torch._lazy_clone(out)                   # shares the memory of `out` until one of them is written
    call(shared)                                      # (a warm call)
    parpy.sync(HIP)
    assert torch.equal(shared, x * 2.0 + b) and bool((out == -1.0).all())
    with pytest.raises(RuntimeError):
        torch.vmap(lambda o: (call(o), o)[1])(torch.zeros(3, 64, device="cuda"))
    call(out)
    assert torch.equal(out, x * 2.0 + b)
