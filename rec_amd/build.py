"""Build recipe for the gfx950 C-ABI library ``rec_amd/librec_amd.so`` and the
Python module ``rec_amd/_host.so`` (the native host path of the small calls).

Run ``python -m rec_amd.build`` (or ``__graft_entry__.build()``).  The
library is compiled in-tree with ``hipcc --offload-arch=gfx950``, the module
with the host compiler against this interpreter's torch; nothing is
JIT-compiled at import time.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "librec_amd.so")
HOST = os.path.join(HERE, "_host.so")
SOURCES = ["abi.hip", "append.hip", "decode.hip", "decode_bf16.hip", "gemv.hip", "q4_gemm.hip", "prefill.hip", "prefill_few.hip"]

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    # keep the compiler from emitting packed-fp32 instructions
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    # MFMA accumulators in ordinary VGPRs: the decode loop rescales them on the
    # VALU, and AGPR accumulators cost a copy out and back per chunk
    "-mllvm",
    "-amdgpu-mfma-vgpr-form",
    "-Wno-unused-command-line-argument",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found: the ROCm toolchain is required to build rec_amd")


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"{os.path.basename(cmd[0])} failed ({proc.returncode}):\n{proc.stderr[-8000:]}")


def _cxx() -> str:
    cxx = os.environ.get("CXX") or shutil.which("g++") or shutil.which("c++")
    if not cxx:
        raise RuntimeError("a C++ compiler is required to build rec_amd/_host.so")
    return cxx


def _host_compile(out: str):
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths

    inc = [f"-I{p}" for p in (*include_paths(), sysconfig.get_paths()["include"])]
    abi = f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}"
    # NDEBUG: without it a torch header's debug counter gives the module
    # thread-local storage, and with glibc before 2.39 loading a module with
    # TLS that nothing touches again sends every other library's TLS access
    # down the slow path (torch.empty 1.5 -> 1.8 us)
    return [_cxx(), "-O2", "-DNDEBUG", "-std=c++17", "-fPIC", "-fvisibility=hidden", abi, *inc,
            "-c", os.path.join(CSRC, "host.cpp"), "-o", out]


def _host_link(libdir: str):
    """Linked to the library beside it (found through $ORIGIN) and to the torch
    libraries an ``import torch`` has mapped."""
    import torch

    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    return [_cxx(), "-shared", "-Wl,--no-as-needed", f"-L{libdir}", f"-L{torch_lib}", "-Wl,-rpath,$ORIGIN",
            "-Wl,--allow-shlib-undefined", "-l:librec_amd.so", "-lc10", "-ltorch_cpu", "-ltorch_python"]


def build(verbose: bool = False, jobs: int = 0) -> str:
    """Compile every HIP source into ``librec_amd.so`` (always rebuilds).

    Each source compiles to its own object (its own device code object) in a
    temporary directory, ``jobs`` at a time (default: one per source, at most
    the CPUs this process may use), then one link makes the library."""
    srcs = [os.path.join(CSRC, s) for s in SOURCES if os.path.exists(os.path.join(CSRC, s))]
    jobs = jobs or max(1, min(len(srcs), len(os.sched_getaffinity(0))))
    compile_flags = [f for f in HIPCC_FLAGS if f != "-shared"]
    with tempfile.TemporaryDirectory(dir=HERE, prefix=".build.") as tmpdir:
        objs = [os.path.join(tmpdir, os.path.basename(s) + ".o") for s in srcs]
        host_obj = os.path.join(tmpdir, "host.o")
        with ThreadPoolExecutor(jobs) as ex:
            host = ex.submit(_run, _host_compile(host_obj), verbose)
            list(ex.map(lambda so: _run([hipcc(), *compile_flags, "-c", so[0], "-o", so[1]], verbose), zip(srcs, objs)))
            host.result()
        tmp = os.path.join(tmpdir, "librec_amd.so")
        _run([hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", tmp], verbose)
        host_tmp = os.path.join(tmpdir, "_host.so")
        _run([*_host_link(tmpdir), host_obj, "-o", host_tmp], verbose)
        os.replace(tmp, LIB)
        os.replace(host_tmp, HOST)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
