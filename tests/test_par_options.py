"""`par`: what it takes and refuses, and that the options hold a copy of the mapping."""
import types

import pytest

import parpy_amd as parpy
from parpy_amd.options import CompileOptions, LoopPar


class Label(str):
    pass


class Par(LoopPar):
    __slots__ = ()


@pytest.mark.parametrize("key,value,ok", [("i", LoopPar(3), True), (Label("i"), LoopPar(3), True), ("i", Par(3), True),
                                          (1, LoopPar(3), False), ("i", 3, False), ("i", None, False)])
def test_labels_and_values(key, value, ok):
    for mapping in ({key: value}, types.MappingProxyType({"j": LoopPar(1), key: value})):
        if not ok:
            with pytest.raises(TypeError):
                parpy.par(mapping)
            continue
        o = parpy.par(mapping)
        assert type(o) is CompileOptions and o.parallelize == dict(mapping) and o.parallelize is not mapping
        assert list(vars(o)) == ["parallelize"]


def test_calls_with_equal_settings_have_equal_keys():
    a, b = (parpy.par({"i": parpy.threads(64).tpb(128), "j": parpy.reduce()}) for _ in range(2))
    assert a._fast_key() == b._fast_key()
    c = parpy.par({"i": parpy.threads(64).tpb(64), "j": parpy.reduce()})
    assert a._fast_key() != c._fast_key()
