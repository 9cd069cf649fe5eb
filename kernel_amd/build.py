"""Compile the HIP sources into ``kernel_amd/libmoe_a2a.so`` for gfx950.

hipcc cross-compiles without a GPU.  Run as ``python -m kernel_amd.build``.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG_DIR)
LIB_PATH = os.path.join(PKG_DIR, "libmoe_a2a.so")
SOURCES = [os.path.join(PKG_DIR, "csrc", "moe_a2a.hip")]

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-ffp-contract=off",  # multiply and add of the weighted sum must stay separate roundings
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",  # no packed-f32 instructions
    "-shared",
    "-fPIC",
    "-I" + os.path.join(ROOT, "include"),
]


def hipcc_path() -> str:
    for cand in (shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (looked on PATH and in /opt/rocm/bin)")


BENCH_LIB_PATH = os.path.join(PKG_DIR, "libmoe_a2a_bench.so")
BENCH_SOURCES = [os.path.join(PKG_DIR, "csrc", "bench_loop.cpp")]


# the host side of the one-call forward: a CPython extension that reads torch's tensor records
HOST_LIB_PATH = os.path.join(PKG_DIR, "_host.so")
HOST_SOURCES = [os.path.join(PKG_DIR, "csrc", "host_path.cpp")]


def _host_command():
    import sysconfig

    import torch
    base = os.path.dirname(os.path.abspath(torch.__file__))
    return ["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-I" + os.path.join(ROOT, "include"),
            "-I" + sysconfig.get_paths()["include"], "-I" + os.path.join(base, "include"),
            "-I" + os.path.join(base, "include", "torch", "csrc", "api", "include"),
            "-I" + os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(hipcc_path()))), "include"),
            *HOST_SOURCES, "-o", HOST_LIB_PATH, "-L" + PKG_DIR, "-lmoe_a2a", "-L" + os.path.join(base, "lib"), "-lc10",
            "-lc10_hip", "-ltorch_cpu", "-ltorch_python", "-Wl,-rpath,$ORIGIN"]


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError("build failed:\n" + proc.stdout + proc.stderr)


def build_library(verbose: bool = False) -> str:
    """The product library, then what links against it: the host extension and the small host-loop helper
    that bench.py uses."""
    _run([hipcc_path(), *HIPCC_FLAGS, *SOURCES, "-o", LIB_PATH], verbose)
    _run(["g++", "-O2", "-shared", "-fPIC", "-I" + os.path.join(ROOT, "include"), *BENCH_SOURCES, "-o",
          BENCH_LIB_PATH, "-L" + PKG_DIR, "-lmoe_a2a", "-Wl,-rpath,$ORIGIN"], verbose)
    _run(_host_command(), verbose)
    return LIB_PATH


if __name__ == "__main__":
    print(build_library(verbose=True))
    sys.exit(0)
