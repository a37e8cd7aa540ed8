"""Builds libmoonep_hip.so (the HIP kernels + C ABI) in-tree for gfx950, and _host.so, the
host side of the Buffer operators (host code against torch's C++ API).

    python -m moonep_amd.build

hipcc cross-compiles without a GPU.  The library sits next to the package so
that it travels with the source tree; nothing is installed.
"""

from __future__ import annotations

import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libmoonep_hip.so")
SOURCES = ["capi.hip", "planner.hip", "dispatch.hip", "combine.hip", "prefetch.hip",
           "grouped_gemm.hip", "gemm_wide.hip"]
GEMM_SOURCES = ["grouped_gemm.hip", "gemm_wide.hip"]    # loads in asm statements, waits counted by hand
FLAGS = [
    "-O3", "-std=c++17", "--offload-arch=gfx950", "-fPIC", "-shared",
    "-Wall", "-Wno-unused-function",
    # packed-fp32 VALU forms are kept off on this hardware pool
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def build_host(verbose: bool = True) -> str:
    """_host.so: no device code, so the host compiler builds it."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths, library_paths

    out = os.path.join(HERE, "_host.so")
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall", "-Wextra",
           "-DUSE_ROCM", "-D__HIP_PLATFORM_AMD__=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *[f"-isystem{p}" for p in (*include_paths("cuda"), sysconfig.get_path("include"))],
           os.path.join(CSRC, "host.cpp"), "-o", out,
           *[f"-L{p}" for p in (*library_paths("cuda"), HERE)],
           "-lmoonep_hip", "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10", "-lc10_hip", "-lamdhip64",
           "-Wl,-rpath,$ORIGIN"]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    return out


def gemm_assembly(out: str, wait: bool = True, source: str = "grouped_gemm.hip"):
    """The compiler's gfx950 assembly of a source of GEMM kernels, with the library's flags."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    cmd = [hipcc, *[f for f in FLAGS if f != "-shared"], "--cuda-device-only", "-S",
           os.path.join(CSRC, source), "-o", out]
    proc = subprocess.Popen(cmd, stderr=subprocess.DEVNULL)      # the library's build shows the warnings
    if wait and proc.wait():
        raise subprocess.CalledProcessError(proc.returncode, cmd)
    return proc


def check_gemm_waits(path: str) -> int:
    """Loads whose waits are counted by hand; raises where the compiler touches one before its wait."""
    from . import asm_waits

    with open(path) as f:
        faults, followed = asm_waits.check(f.read())
    if faults or not followed:
        raise RuntimeError("the GEMM kernels as this compiler builds them are not safe to run: " +
                           ("; ".join(faults[:8]) or "no load in an asm statement was found"))
    return followed


def build(verbose: bool = True) -> str:
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    cmd = [hipcc, *FLAGS, *[os.path.join(CSRC, s) for s in SOURCES], "-o", LIB]
    if verbose:
        print(" ".join(cmd), flush=True)
    with tempfile.TemporaryDirectory() as tmp:
        beside = []
        for source in GEMM_SOURCES:
            path = os.path.join(tmp, source + ".s")
            beside.append((path, gemm_assembly(path, wait=False, source=source)))
        try:
            subprocess.run(cmd, check=True)
        finally:
            failed = [proc for _, proc in beside if proc.wait()]
        if failed:
            raise subprocess.CalledProcessError(failed[0].returncode, failed[0].args)
        try:
            for path, _ in beside:
                check_gemm_waits(path)
        except RuntimeError:
            os.remove(LIB)
            raise
    build_host(verbose)
    return LIB


if __name__ == "__main__":
    build()
    sys.exit(0)
