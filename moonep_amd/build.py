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

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libmoonep_hip.so")
SOURCES = ["capi.hip", "planner.hip", "dispatch.hip", "combine.hip", "prefetch.hip",
           "grouped_gemm.hip"]
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
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-w",
           "-DUSE_ROCM", "-D__HIP_PLATFORM_AMD__=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *[f"-I{p}" for p in (*include_paths("cuda"), sysconfig.get_path("include"))],
           os.path.join(CSRC, "host.cpp"), "-o", out,
           *[f"-L{p}" for p in (*library_paths("cuda"), HERE)],
           "-lmoonep_hip", "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10", "-lc10_hip", "-lamdhip64",
           "-Wl,-rpath,$ORIGIN"]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    return out


def build(verbose: bool = True) -> str:
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    cmd = [hipcc, *FLAGS, *[os.path.join(CSRC, s) for s in SOURCES], "-o", LIB]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    build_host(verbose)
    return LIB


if __name__ == "__main__":
    build()
    sys.exit(0)
