"""Build libaar_hip.so in-tree with hipcc for gfx950.

    python linear-solver_amd/aar_hip/build.py

Objects are compiled in parallel into linear-solver_amd/_build/ and linked
into linear-solver_amd/libaar_hip.so, which the ctypes loader picks up.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

PKG_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))   # linear-solver_amd/
REPO = os.path.dirname(PKG_ROOT)
CSRC = os.path.join(PKG_ROOT, "csrc")
INCLUDE = os.path.join(REPO, "include")
BUILD = os.path.join(PKG_ROOT, "_build")
LIB = os.path.join(PKG_ROOT, "libaar_hip.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("AAR_HIP_ARCH", "gfx950")

SOURCES = ["stencil.hip", "stencil_vc.hip", "history.hip", "ls.hip", "update.hip", "helmholtz.hip", "batch.hip",
           "solver.hip", "krylov.hip", "ilu.hip", "capi.hip", "stream.hip", "noalloc.hip"]

# -ffp-contract=off: the stencil, the Richardson/Anderson updates and the
# SVD must not fuse multiply-adds, so that they round exactly as the
# reference's FMA-free x86-64 build does.  Packed FP32 is disabled.
# -falign-loops=64: the march's plane loop starts on an instruction fetch line
# wherever it lands in its kernel (512^3 FP64 recurrence 424-426 us, 432 with the
# same instructions elsewhere).
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-fPIC", "-std=c++17", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-falign-loops=64",
    "-I" + INCLUDE, "-I" + CSRC,
]


def _compile(src):
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC] + FLAGS + ["-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr[-4000:]}")
    return obj


def build(verbose=True):
    os.makedirs(BUILD, exist_ok=True)
    with ThreadPoolExecutor(max_workers=min(8, len(SOURCES))) as ex:
        objs = list(ex.map(_compile, SOURCES))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr[-4000:]}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build()
    sys.exit(0)
