"""Loader of the extension that serves warm calls (csrc/runtime/fastcall.cpp -> _fastcall.so).

The extension reads torch tensors through torch's own headers, so it is built against the torch that is installed, by
`__graft_entry__.build()`; a library that does not match its source is rebuilt when it is first needed, as with the
other native parts.  Calls run without it too, only slower: on a machine without torch there is nothing to serve, where
it can neither be loaded nor built a warning says why, once, and `call_table` returns None in both cases.
"""
import ctypes
import importlib.machinery
import importlib.util
import os
import pathlib
import subprocess
import sys
import sysconfig
import warnings

from . import _buildstamp

SOURCE = pathlib.Path(__file__).parent / "csrc" / "runtime" / "fastcall.cpp"
LIB_PATH = pathlib.Path(__file__).parent / "_fastcall.so"

_module = None
_unavailable = False   # neither loaded nor built: not tried again in this process


def _command():
    import torch
    return ["g++", "-std=c++17", "-O2", "-fPIC", "-shared", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
            "-D__HIP_PLATFORM_AMD__=1", f"-I{sysconfig.get_paths()['include']}"]


def _stamped():
    """What the library is built with and against.  The folders of torch's headers and libraries follow from its version
    and place; the module that lists them takes 0.2 s to import and is left to the builds."""
    import torch
    return _command() + [f"torch-{torch.__version__}", os.path.dirname(torch.__file__)]


def build_library(force=False):
    """Compile the extension with g++ (no GPU toolchain needed)."""
    cmd = _stamped()
    if not force and LIB_PATH.exists() and _buildstamp.is_current(LIB_PATH, [SOURCE], cmd):
        return LIB_PATH
    from torch.utils.cpp_extension import include_paths, library_paths
    paths = [f"-isystem{p}" for p in include_paths()] + [x for p in library_paths() for x in (f"-L{p}", f"-Wl,-rpath,{p}")]
    tmp = LIB_PATH.with_suffix(f".tmp{os.getpid()}")
    r = subprocess.run(_command() + paths + ["-o", str(tmp), str(SOURCE), "-ltorch_python", "-ltorch_cpu", "-lc10"], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"Compilation of the call extension failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB_PATH)
    _buildstamp.write_stamp(LIB_PATH, [SOURCE], cmd)
    return LIB_PATH


def _load():
    global _module
    if _module is None:
        _buildstamp.ensure_current(LIB_PATH, [SOURCE], _stamped(), lambda: build_library(force=True))
        loader = importlib.machinery.ExtensionFileLoader("_fastcall", str(LIB_PATH))
        spec = importlib.util.spec_from_file_location("_fastcall", str(LIB_PATH), loader=loader)
        _module = importlib.util.module_from_spec(spec)
        loader.exec_module(_module)
    return _module


def call_table(lib):
    """A table of warm calls that run plans of the runtime library `lib`; None where the extension cannot be had.  It is
    asked for when the first call has run, which must not fail for it any more."""
    global _unavailable
    if "torch" not in sys.modules or _unavailable:
        return None
    from .options import CompileOptions, LoopPar
    try:
        module = _load()
    except Exception as e:
        _unavailable = True
        warnings.warn(f"Warm calls take the slower Python path, their extension {LIB_PATH.name} cannot be had: {e}", RuntimeWarning)
        return None
    return module.CallTable(CompileOptions, LoopPar, ctypes.cast(lib.parpy_hip_plan_run, ctypes.c_void_p).value)


def pointer_order(args):
    """order[k]: which of the call's array tensors, counted as they stand in the arguments, is pointer k of the plan
    (dictionary fields are passed sorted by key)."""
    torch = sys.modules["torch"]
    is_array = lambda v: type(v) is torch.Tensor and v.dim() > 0
    order, base = [], 0
    for a in args:
        if type(a) is dict:
            names = [k for k, v in a.items() if is_array(v)]
            at = {k: base + i for i, k in enumerate(names)}
            order += [at[k] for k in sorted(names)]
            base += len(names)
        elif is_array(a):
            order.append(base)
            base += 1
    return tuple(order)
