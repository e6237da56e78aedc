"""Build libfwiflow_hip.so for gfx950 (hipcc for the kernels, g++ for host code).

Usage: python fwiflow.jl_amd/build.py   (always recompiles).
Objects go to fwiflow.jl_amd/_build/, the library to fwiflow.jl_amd/lib/.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "_build")
LIBDIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIBDIR, "libfwiflow_hip.so")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
HIPCC = os.path.join(ROCM, "bin", "hipcc")
ARCH = "gfx950"

HOST_SRC = ["json.cpp", "config.cpp", "capi.cpp"]
HIP_SRC = ["engine.hip", "cnn.hip", "cond.hip"]

CXXFLAGS = ["-O2", "-std=c++17", "-fPIC", "-Wall", "-Wextra", "-Wno-unused-parameter"]
# packed-FP32 instructions are disabled for all device code.  Multiply-add
# contraction is limited to single source expressions (-ffp-contract=on), so
# the rounding of a stencil update depends on how it is written, not on the
# kernel it is inlined into: the one-launch and two-launch forms of
# a step then agree to the last bit wherever they share an expression.
# The first 16 words of a kernel's arguments arrive in scalar registers: a
# workgroup of a short launch otherwise waits for them first (one of the 3.6 us
# of a 64x84 step; 5% of that modelling run, 3-4% of 164x264 and 127x341
# gradients, 1% at 580x1780).
HIPFLAGS = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-Wall",
            "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
            "-ffp-contract=on", "-munsafe-fp-atomics",
            "-mllvm", "-amdgpu-kernarg-preload-count=16"]
# extra compiler definitions for A/B builds of engine switches (space separated)
HIPFLAGS += os.environ.get("FWIFLOW_HIPFLAGS", "").split()


def _run(cmd):
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(" ".join(cmd) + "\n" + r.stdout + r.stderr)
        raise RuntimeError(f"build step failed: {cmd[0]} {cmd[-1]}")
    return r


def build(verbose: bool = False) -> str:
    os.makedirs(OBJ, exist_ok=True)
    os.makedirs(LIBDIR, exist_ok=True)
    jobs = []
    for s in HOST_SRC:
        o = os.path.join(OBJ, s + ".o")
        jobs.append(["g++", *CXXFLAGS, "-c", os.path.join(CSRC, s), "-o", o])
    for s in HIP_SRC:
        o = os.path.join(OBJ, s + ".o")
        jobs.append([HIPCC, *HIPFLAGS, "-c", os.path.join(CSRC, s), "-o", o])
    with ThreadPoolExecutor(max_workers=4) as ex:
        for r in ex.map(_run, jobs):
            if verbose and (r.stdout or r.stderr):
                print(r.stdout + r.stderr)
    objs = [j[-1] for j in jobs]
    tmp = LIB + ".tmp"
    _run([HIPCC, "-shared", f"--offload-arch={ARCH}", "-o", tmp, *objs,
          f"-Wl,-rpath,{ROCM}/lib"])
    shutil.move(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
