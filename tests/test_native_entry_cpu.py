"""The C++ entry of the launch-bound operators (csrc/native.cpp) on the CPU: a
copy of the built module, bound to host stand-ins of the C ABI's functions, so
that what happens around a launch can be looked at without one."""
from __future__ import annotations

import ctypes
import importlib
import importlib.util
import shutil
import subprocess
import sys
import threading
import types

import pytest
import torch

import spikeinfer_amd
from spikeinfer_amd import _lib
from spikeinfer_amd.build import NATIVE_PATH


ERROR = ctypes.create_string_buffer(b"the stand-in's error")
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
        default = lambda *a: 0
        if name == "spk_last_error":
            res, default = ctypes.c_void_p, lambda: ctypes.addressof(ERROR)
        fn = ctypes.CFUNCTYPE(res, *args)(stubs.get(name, default))
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


def _calls(n=64):
    """Each operator's name in the module, its C function and arguments it takes."""
    f, b16 = torch.float32, torch.bfloat16
    z = lambda *s, dt=f: torch.zeros(s, dtype=dt)
    i32, i64 = torch.int32, torch.int64
    q, kv = z(4, 2, 4, 2, dt=i32), z(4, 2, 32, 2, dt=i32)
    lens, table = torch.ones(2, dtype=i32), z(2, 2, dt=i32)
    h, w = z(4, 3, n, dt=b16), z(n, dt=b16)
    qkv, rope = z(4, 2, 8 * 64, dt=b16), z(5, 64, dt=b16)
    slots = torch.arange(2)
    return [
        ("decode_attn", "spk_decode_attn", (q, kv, kv, table, lens, 64, 16, 4, 2, None, f, None)),
        ("lif_sites", "spk_lif_pack_write_sites", ([(z(4, 2, 4, 64), z(64), z(64), q, False)], None)),
        ("lif", "spk_lif_multistep", (z(4, 3, n), z(n), z(n), True)),
        ("prefill", "spk_prefill_attn", (q, kv, kv, [(0, 0, 2, 1, table[0])], z(4, 2, 4, 64), 64, 16)),
        ("embed_rmsnorm", "spk_embed_rmsnorm", (z(3, dt=i64), z(9, n, dt=b16), w, 1e-6, 4)),
        ("add_rmsnorm", "spk_add_rmsnorm", (h, torch.ones_like(h), w, 1e-6, None)),
        ("rmsnorm_mean_t", "spk_rmsnorm_mean_t", (h, w, 1e-6, None)),
        ("lif_gate_mul", "spk_lif_gate_mul", (h, z(n // 2), z(n // 2))),
        ("linear_decode", "spk_linear_decode", (h, z(16, n, dt=b16), None, None)),
        ("mlp_gate_lif", "spk_mlp_gate_lif", (h, z(2 * 32, n, dt=b16), z(32), z(32))),
        ("qkv_rope_lif_pack", "spk_qkv_rope_lif_pack_kv", (qkv, rope, rope, z(3, 64), z(3, 64), kv, kv, slots, 4, 2,
                                                           64, q, 2, slots, None, None)),
    ]


@pytest.mark.parametrize("status", [_lib.SPK_OK, _lib.SPK_EINVAL, _lib.SPK_EUNSUPPORTED, _lib.SPK_EHIP])
def test_a_call_is_repeated_only_if_nothing_was_launched(tmp_path, status):
    """Refusals (decided before a launch) go back to the wrapper; an error read after
    the launch is raised, so that nothing runs twice."""
    for name, fn, args in _calls():
        (tmp_path / name).mkdir()
        seen = []
        mod = load_with_stubs(tmp_path / name, **{fn: lambda *a: seen.append(a) or status})
        call = getattr(mod, name)
        if status == _lib.SPK_EHIP:
            with pytest.raises(RuntimeError, match="the stand-in's error"):
                call(*args)
        else:
            assert (call(*args) is None) == (status != _lib.SPK_OK), name
        assert len(seen) == 1, name


def test_the_residual_is_added_once(tmp_path, monkeypatch):
    """add_rmsnorm updates h in place: through the wrapper, an error that is read
    after the launch leaves one launch behind it and reaches the caller."""
    from spikeinfer_amd.kernels.decoder_ops import add_rmsnorm

    h, delta = torch.zeros(2, 8), torch.ones(2, 8)
    seen = []

    def launched(*a):
        seen.append(h.add_(delta))
        return _lib.SPK_EHIP if len(seen) == 1 else _lib.SPK_OK

    monkeypatch.setattr(_lib, "_native", load_with_stubs(tmp_path, spk_add_rmsnorm=launched))
    monkeypatch.setattr(_lib, "require_gpu", lambda *t: torch.device("cpu"))
    monkeypatch.setattr(_lib, "stream_of", lambda d: 0)
    host = type("Host", (), {"spk_add_rmsnorm": staticmethod(launched)})
    monkeypatch.setattr(_lib, "load", lambda path=None: host)
    with pytest.raises(RuntimeError, match="add_rmsnorm: the stand-in's error"):
        add_rmsnorm(h, delta, torch.ones(8), 1e-6)
    assert len(seen) == 1 and torch.equal(h, delta)


def test_rows_past_64_bits_are_not_taken(tmp_path):
    """A chunk's first row near 2**63: the row after its last must not wrap round to
    one inside the tensor."""
    seen = []
    mod = load_with_stubs(tmp_path, spk_prefill_attn=lambda *a: seen.append(a) or 0)
    args = dict((name, a) for name, _, a in _calls())["prefill"]
    for q_row, out_row in ((2**63 - 1, 0), (2**63 - 2, 2**63 - 2), (0, 2**63 - 1), (-1, 0), (1, 0), (0, 1)):
        assert mod.prefill(*args[:3], [(q_row, out_row, 2, 0, args[3][0][4])], *args[4:]) is None
    assert not seen
    assert mod.prefill(*args) is True and len(seen) == 1


def _fresh(monkeypatch, module):
    """_lib.native() as a new process would answer it with `module` beside it."""
    monkeypatch.setattr(_lib, "_native", _lib._UNBOUND)
    monkeypatch.setitem(sys.modules, "spikeinfer_amd._native", module)
    monkeypatch.setattr(spikeinfer_amd, "_native", module, raising=False)
    return _lib.native()


def test_a_module_built_for_something_else_is_not_used(monkeypatch):
    """Its calls go to bare addresses: another version of the C ABI or of torch
    than it was compiled for means the wrappers' own path."""
    binds = []
    stamp = dict(abi_version=_lib.ABI_VERSION, built_for=torch.__version__)
    for change, used in ((dict(), True), (dict(abi_version=3), False), (dict(built_for="2.0.0"), False),
                         (dict(abi_version=None, built_for=None), False)):
        mod = types.ModuleType("_native")
        mod.bind = lambda *a: binds.append(a)
        for name, value in {**stamp, **change}.items():
            if value is not None:
                setattr(mod, name, value)
        assert _fresh(monkeypatch, mod) is (mod if used else None), change
    assert len(binds) == 1


def test_the_built_module_is_stamped_and_used(monkeypatch):
    mod = importlib.import_module("spikeinfer_amd._native")
    assert (mod.abi_version, mod.built_for) == (_lib.ABI_VERSION, torch.__version__)
    assert _fresh(monkeypatch, mod) is mod
