"""Builds libspikeinfer_amd.so (gfx950) in-tree with hipcc, and _native.so (the
Python entry of the launch-bound operators) with g++.

Usage: ``python -m spikeinfer_amd.build`` (or ``build()`` from Python).  The
library is a plain C-ABI shared object (see include/spikeinfer_amd.h); it is
loaded with ctypes by ``spikeinfer_amd._lib``.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_NAME = "libspikeinfer_amd.so"
LIB_PATH = os.path.join(HERE, LIB_NAME)
ARCH = "gfx950"

# -ffp-contract=off: the LIF recurrence must round mul and add separately.
# -packed-fp32-ops off: no v_pk_*_f32 in generated code.
HIPCC_FLAGS = [
    "-O3", "-std=c++17", "-fPIC",
    f"--offload-arch={ARCH}",
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def sources() -> list[str]:
    return sorted(
        os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip")
    )


OBJ_DIR = os.path.join(HERE, "_build")
NATIVE_PATH = os.path.join(HERE, "_native.so")


def native_command(out: str) -> list[str]:
    """The g++ line of the Python entry (csrc/native.cpp) against the installed torch."""
    import sysconfig

    import torch

    root = os.path.dirname(torch.__file__)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    includes = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
                os.path.join(rocm, "include"), sysconfig.get_paths()["include"]]
    return [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1",
            "-DUSE_ROCM=1", f'-DSPK_TORCH_VERSION="{torch.__version__}"',
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
            *(f"-I{i}" for i in includes), "-o", out, os.path.join(CSRC, "native.cpp"),
            "-L" + os.path.join(root, "lib"), "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python"]


def _run(cmd: list[str], verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{os.path.basename(cmd[0])} failed ({res.returncode}):\n{res.stderr}")


def build_native(verbose: bool = False) -> str | None:
    """Compiles csrc/native.cpp into the Python entry module; what failed, if it
    did (an older module is then removed: it may be of another C ABI)."""
    tmp = NATIVE_PATH + ".tmp"
    try:
        _run(native_command(tmp), verbose)
        os.replace(tmp, NATIVE_PATH)
        return None
    except Exception as e:  # no compiler, no headers of torch or Python, a compile error
        if os.path.exists(NATIVE_PATH):
            os.remove(NATIVE_PATH)
        return str(e)


def build(verbose: bool = False) -> str:
    """Compiles every csrc/*.hip to an object (in parallel, one hipcc per
    file) and links them into the shared library, and csrc/native.cpp into
    the Python entry module beside it.  Always recompiles.  Without the entry
    module the operators make their calls through ctypes, so a failure there
    is a warning on stderr."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs = sources()
    objs = [os.path.join(OBJ_DIR, os.path.basename(s)[:-4] + ".o") for s in srcs]
    jobs = max(1, min(len(srcs) + 1, os.cpu_count() or 1, 16))
    with ThreadPoolExecutor(jobs) as ex:
        native = ex.submit(build_native, verbose)
        list(ex.map(lambda so: _run([hipcc, *HIPCC_FLAGS, "-c", "-o", so[1], so[0]], verbose),
                    zip(srcs, objs)))
        failed = native.result()
    tmp = LIB_PATH + ".tmp"
    _run([hipcc, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", tmp, *objs], verbose)
    os.replace(tmp, LIB_PATH)
    if failed:
        print(f"warning: {NATIVE_PATH} not built, calls go through ctypes: {failed}", file=sys.stderr)
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
