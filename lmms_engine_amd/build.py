"""Builds lmms_engine_amd/libmuon_hip.so from csrc/ with hipcc for gfx950, and the host-side Python module _scan beside it.

Run as `python -m lmms_engine_amd.build` or call build_library().  The library is built
in-tree, next to this file, so it travels with the source tree.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libmuon_hip.so")
SOURCES = ["gemm_nt.hip", "elementwise.hip", "small_chain.hip", "multi_tensor.hip", "api.hip"]
# Measurement kernels (MFMA-only loops) for the benchmark's operand-power legs: a library of their own, no part of the product.
PROBE_LIB = os.path.join(HERE, "libmuon_probe.so")
PROBE_SOURCES = ["probe.hip"]
# Reads lists of torch tensors for the optimizer step (host code; a Python module, since it handles Python objects).  Its name says
# which Python it is for, and it carries the version of the torch whose headers it was compiled with (checked when it is loaded).
SCAN_LIB = os.path.join(HERE, "_scan" + sysconfig.get_config_var("EXT_SUFFIX"))
# Packed-fp32 VALU forms stay off for every device function.
HIP_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-fPIC",
    "-std=c++17",
    "-fvisibility=hidden",  # the libraries export their extern "C" entry points and nothing else
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _compile_and_link(sources, lib, hipcc, verbose):
    objdir = os.path.join(CSRC, "build")
    os.makedirs(objdir, exist_ok=True)
    procs = []
    for src in sources:
        obj = os.path.join(objdir, src.replace(".hip", ".o"))
        cmd = [hipcc, *HIP_FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((src, obj, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
    objs = []
    for src, obj, p in procs:
        out, _ = p.communicate()
        out = "\n".join(l for l in out.splitlines() if "not a recognized feature" not in l)
        if p.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src}:\n{out}")
        if verbose and out.strip():
            print(out)
        objs.append(obj)
    cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", lib]
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}")
    return lib


def _build_scan(verbose):
    import torch
    from torch.utils.cpp_extension import include_paths, library_paths

    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f'-DSCAN_TORCH_VERSION="{torch.__version__}"', *[f"-isystem{p}" for p in include_paths()], f"-isystem{sysconfig.get_paths()['include']}", os.path.join(CSRC, "scan.cpp"), "-o", SCAN_LIB,
           *[f"-L{p}" for p in library_paths()], "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10"]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed on scan.cpp:\n{r.stdout}")


def built() -> bool:
    """Whether everything that the package loads is there."""
    return os.path.exists(LIB) and os.path.exists(SCAN_LIB)


def build_library(verbose: bool = False) -> str:
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        raise RuntimeError("hipcc not found; cannot build libmuon_hip.so")
    _build_scan(verbose)
    _compile_and_link(PROBE_SOURCES, PROBE_LIB, hipcc, verbose)
    return _compile_and_link(SOURCES, LIB, hipcc, verbose)


if __name__ == "__main__":
    print(build_library(verbose="-v" in sys.argv))
