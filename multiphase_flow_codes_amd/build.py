"""Builds libmfc_lbm.so (HIP, gfx950) in-tree with hipcc.

``python -m multiphase_flow_codes_amd.build`` or ``build_library()``.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libmfc_lbm.so")
ARCH = os.environ.get("MFC_OFFLOAD_ARCH", "gfx950")

COMMON = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
    # no packed-FP32 instructions in device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-variable",
]
# per-source extra flags: the particle geometry is evaluated without
# floating-point contraction so node maps match the FP64 reference exactly;
# the lattice kernels contract a*b+c only within one source expression, so
# every kernel variant that shares the collision code (two buffers, in place,
# batched) rounds it identically whatever code surrounds it
SOURCES = {
    "api.hip": [],
    "fluid.hip": ["-ffp-contract=on"],
    "particles.hip": ["-ffp-contract=off"],
    "diag.hip": [],
    "ensemble.hip": [],
    "initial.hip": [],
    "hostcopy.hip": [],
}


def _run(cmd):
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(" ".join(cmd) + "\n" + r.stdout + r.stderr)
        raise RuntimeError(f"hipcc failed ({r.returncode}) on {cmd[-1]}")
    return r


def build_library(verbose: bool = False) -> str:
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    objdir = os.path.join(HERE, "_build")
    os.makedirs(objdir, exist_ok=True)
    cmds, objs = [], []
    for src, extra in SOURCES.items():
        obj = os.path.join(objdir, src.replace(".hip", ".o"))
        cmds.append([hipcc, *COMMON, *extra, "-c", "-o", obj, os.path.join(CSRC, src)])
        objs.append(obj)
        if verbose:
            print(" ".join(cmds[-1]), flush=True)
    jobs = max(1, min(len(cmds), int(os.environ.get("MAX_JOBS", "4"))))
    with ThreadPoolExecutor(jobs) as pool:
        list(pool.map(_run, cmds))
    tmp = LIB + ".tmp"
    _run([hipcc, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", tmp, *objs])
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build_library(verbose=True))
