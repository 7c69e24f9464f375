"""The C++ entry of the launch-bound operators (csrc/native.cpp) on the CPU: a
copy of the built module, bound to host stand-ins of the C ABI's functions, so
that what happens around a launch can be looked at without one."""
from __future__ import annotations

import ctypes
import importlib.util
import shutil
import subprocess
import sys
import threading

import pytest
import torch

from spikeinfer_amd import _lib
from spikeinfer_amd.build import NATIVE_PATH


bound = {}  # module file -> its stand-ins, which it calls as long as it lives


def load_with_stubs(folder, **stubs):
    """A module of its own (its globals are per file), bound to `stubs`: name ->
    Python function of the C function's arguments.  The others return SPK_OK."""
    path = shutil.copy(NATIVE_PATH, folder)
    spec = importlib.util.spec_from_file_location("_native", path)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    addresses, keep = [], []
    for name in _lib.NATIVE_FUNCTIONS:
        res, args = _lib._SIGNATURES[name]
        # (pointers as plain addresses: a callback gets no typed pointer from C)
        args = [ctypes.c_void_p if a not in (ctypes.c_int, ctypes.c_int64, ctypes.c_float, ctypes.c_size_t) else a
                for a in args]
        fn = ctypes.CFUNCTYPE(res, *args)(stubs.get(name, lambda *a: 0))
        keep.append(fn)
        addresses.append(ctypes.cast(fn, ctypes.c_void_p).value)
    mod.bind("cpu", *addresses)
    bound[path] = keep
    return mod


def test_tensors_without_storage_are_not_taken(tmp_path):
    """Inside torch.vmap and torch.func.grad an argument is a plain torch.Tensor
    without storage: the call goes back to the wrapper, which raises.  In a
    process of its own, so that a crash is a failure."""
    code = f"""
import sys, torch
sys.path[:0] = {sys.path!r}
from test_native_entry_cpu import load_with_stubs
calls = []
mod = load_with_stubs({str(tmp_path)!r}, spk_lif_multistep=lambda *a: calls.append(a) or 0)
b, th = torch.full((8,), 0.9), torch.ones(8)
assert mod.lif(torch.zeros(4, 3, 8), b, th, False).shape == (4, 3, 8) and len(calls) == 1
def f(x):
    assert mod.lif(x, b, th, False) is None
    assert mod.add_rmsnorm(x, None, b, 1e-6, None) is None
    return x.sum()
torch.vmap(f)(torch.zeros(2, 4, 3, 8))
torch.func.grad(f)(torch.zeros(4, 3, 8))
assert len(calls) == 1
"""
    done = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, (done.returncode, done.stderr[-2000:])


def test_the_interpreter_is_free_during_a_launch(tmp_path):
    """Two threads inside launches at once: each waits for the other in the
    stand-in, which itself needs the interpreter."""
    meet = threading.Barrier(2, timeout=60)
    mod = load_with_stubs(tmp_path, spk_lif_multistep=lambda *a: int(meet.wait() < 0))
    args = torch.zeros(4, 3, 8), torch.full((8,), 0.9), torch.ones(8)
    got = [None, None]

    def work(i):
        got[i] = mod.lif(*args, False)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(120)
    assert all(g is not None and g.shape == (4, 3, 8) for g in got)
