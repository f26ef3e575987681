"""`threads` and `par` of the extension: what they make is what the Python functions make, and what they do not take plainly is
left to those."""
import inspect
import pickle
import types

import pytest

import parpy_amd as parpy
from parpy_amd import fastopts
from parpy_amd.options import CompileOptions, LoopPar


class Count(int):
    pass


class Par(LoopPar):
    __slots__ = ()


class Mapping(dict):
    pass


def test_the_extension_is_the_one_that_runs():
    assert type(parpy.threads) is type(parpy.par) is types.BuiltinFunctionType and parpy.options.par is parpy.par
    for f in (parpy.threads, parpy.par):
        assert pickle.loads(pickle.dumps(f)) is f and f.__doc__ and len(inspect.signature(f).parameters) == 1


@pytest.mark.parametrize("n", [0, 1, 5, -3, 1 << 70, True, Count(7), 2.5, "12"])
def test_threads(n):
    for p in (parpy.threads(n), parpy.threads(n=n)):
        assert type(p) is LoopPar and type(p.nthreads) is int and p.nthreads == int(n) and p.reduction is False and p == LoopPar(int(n))
    p, q = parpy.threads(n), parpy.threads(n)
    p.nthreads = 9
    assert q.nthreads == int(n) and repr(q.tpb(128)) == repr(LoopPar(int(n)).tpb(128))


def test_what_threads_refuses():
    for args, kw, error in [((), {}, TypeError), ((1, 2), {}, TypeError), ((1,), {"n": 1}, TypeError), ((None,), {}, TypeError), (("x",), {}, ValueError)]:
        with pytest.raises(error):
            parpy.threads(*args, **kw)


@pytest.mark.parametrize("mapping", [{}, {"i": LoopPar(3)}, {"i": LoopPar(3), "j": LoopPar(0).reduce()}, Mapping(i=LoopPar(3)), {"i": Par(3)}])
def test_par(mapping):
    before = dict(mapping)
    for o in (parpy.par(mapping), parpy.par(p=mapping)):
        assert type(o) is CompileOptions and list(vars(o)) == ["parallelize"] and type(o.parallelize) is dict and o.parallelize is not mapping
        o.parallelize["k"] = LoopPar(1)
        assert mapping == before
    for args in ((), (1,), ({"i": 3},), ({1: LoopPar(3)},), ({}, {})):
        with pytest.raises((TypeError, AttributeError)):
            parpy.par(*args)


def test_nothing_is_kept_or_lost():
    import sys
    n, mapping = 123456789, {"i": LoopPar(3)}
    counts = [sys.getrefcount(x) for x in (n, mapping["i"], LoopPar, CompileOptions)]
    for _ in range(1000):
        parpy.threads(n), parpy.par(mapping)
        for bad in (lambda: parpy.threads(None), lambda: parpy.par({"i": 3})):
            with pytest.raises(TypeError):
                bad()
    assert all(abs(a - sys.getrefcount(x)) <= 2 for a, x in zip(counts, (n, mapping["i"], LoopPar, CompileOptions)))


def test_without_the_extension_the_python_functions_stay(monkeypatch):
    def missing(*a, **k):
        raise OSError("no compiler")
    monkeypatch.setattr(fastopts._buildstamp, "ensure_current", missing)
    threads, par = object(), object()
    assert fastopts.faster(LoopPar, 1024, CompileOptions, threads, par) == (threads, par)


def test_without_the_extension(monkeypatch):
    """A folder that cannot be written: no compiler is started, the functions stay as they are and a warning says so."""
    functions = object(), object()
    monkeypatch.setattr(fastopts.os, "access", lambda path, mode: False)
    monkeypatch.setattr(fastopts._buildstamp, "is_current", lambda *args: False)
    monkeypatch.setattr(fastopts.subprocess, "run", lambda *args, **kw: pytest.fail("a compiler was started"))
    with pytest.warns(RuntimeWarning, match="cannot be written"):
        assert fastopts.faster(LoopPar, 1024, CompileOptions, *functions) == functions
