"""Loader of the extension that builds the options of a call (csrc/runtime/fastopts.c -> _fastopts.so).

Built by `__graft_entry__.build()`; a library that does not match its source is rebuilt when the package is imported, as
with the other native parts when they are needed, if its folder can be written.  Where it cannot be had the Python functions stay,
which do the same, a third of a microsecond slower, and a warning says why.
"""
import importlib.machinery
import importlib.util
import os
import pathlib
import subprocess
import sysconfig
import warnings

from . import _buildstamp

SOURCE = pathlib.Path(__file__).parent / "csrc" / "runtime" / "fastopts.c"
LIB_PATH = pathlib.Path(__file__).parent / "_fastopts.so"


def _command():
    return ["gcc", "-std=c11", "-O2", "-fPIC", "-shared", f"-I{sysconfig.get_paths()['include']}"]


def build_library(force=False):
    cmd = _command()
    if not force and LIB_PATH.exists() and _buildstamp.is_current(LIB_PATH, [SOURCE], cmd):
        return LIB_PATH
    tmp = LIB_PATH.with_suffix(f".tmp{os.getpid()}")
    r = subprocess.run(cmd + ["-o", str(tmp), str(SOURCE)], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"Compilation of the options extension failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB_PATH)
    _buildstamp.write_stamp(LIB_PATH, [SOURCE], cmd)
    return LIB_PATH


def faster(loop_par, tpb, options, threads, par):
    """`threads` and `par` as functions of the extension, or as they are."""
    try:
        # (an installation that cannot be written does not start a compiler in every import)
        if not os.access(LIB_PATH.parent, os.W_OK) and not _buildstamp.is_current(LIB_PATH, [SOURCE], _command()):
            raise RuntimeError("it is not there or does not match its source, and its folder cannot be written")
        _buildstamp.ensure_current(LIB_PATH, [SOURCE], _command(), lambda: build_library(force=True))
        loader = importlib.machinery.ExtensionFileLoader("_fastopts", str(LIB_PATH))
        module = importlib.util.module_from_spec(importlib.util.spec_from_file_location("_fastopts", str(LIB_PATH), loader=loader))
        loader.exec_module(module)
        return module.functions(loop_par, tpb, options, threads, par)
    except Exception as e:
        warnings.warn(f"Options of a call are made by the slower Python functions, their extension {LIB_PATH.name} cannot be had: {e}", RuntimeWarning)
        return threads, par
