"""Builds kata_amd/libkata_amd.so (gfx950) in-tree with hipcc.

    python -m kata_amd.build        # or kata_amd.build.build()

Every HIP source is compiled for gfx950 only, with packed-fp32 instruction generation
disabled on the device side, then linked into one shared library exporting the C ABI of
include/kata_amd.h.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libkata_amd.so")
SOURCES = ["gemv_ptq1.hip", "gemv_q8.hip", "gemm_f16.hip", "gemm_q8.hip", "gemm_i8.hip", "expand.hip", "norm_fwht.hip", "argmax.hip", "calib.hip", "workspace.cpp", "gguf.cpp", "capi.cpp"]
# Per-source extra flags.  The fp16 and Q8_0 prefill GEMMs keep up to 256 fp32 accumulators per
# lane beside their decode code; LLVM's iterative-ILP scheduler keeps them in place (the default
# one shuttles them between register files every stage).  The GEMV and int8 GEMM sources take the
# max-ILP scheduler (decode sweep step 45.1 -> 44.7 us, wide T = 8 gate 10.5 -> 10.3 us;
# int8 gate / down at 512 rows 88.1 / 81.7 -> 86.6 / 79.7 us; results unchanged).  Measured and
# left at the default: the Q8_0 GEMV (max-ILP slower; iterative-ILP 21.2 -> 31.9 us on
# 5120 x 17408) and the input transform (no change).
EXTRA_FLAGS = {"gemm_f16.hip": ["-mllvm", "-amdgpu-sched-strategy=iterative-ilp"],
               "gemm_q8.hip": ["-mllvm", "-amdgpu-sched-strategy=iterative-ilp"],
               "gemv_ptq1.hip": ["-mllvm", "-amdgpu-sched-strategy=max-ilp"],
               "gemm_i8.hip": ["-mllvm", "-amdgpu-sched-strategy=max-ilp"]}
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "-O3", "-std=c++17", "-fPIC", "--offload-arch=gfx950",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]


def _compile(src: str) -> str:
    obj = os.path.join(OBJ, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC, "-x", "hip", *FLAGS, *EXTRA_FLAGS.get(src, []), "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr}")
    # the host-side cc1 does not know the device feature; every other warning is shown
    noise = "'-packed-fp32-ops' is not a recognized feature"
    warn = "\n".join(l for l in r.stderr.splitlines() if noise not in l)
    if warn.strip():
        print(warn, file=sys.stderr)
    return obj


def build(verbose: bool = True) -> str:
    os.makedirs(OBJ, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=min(8, len(SOURCES))) as ex:
        objs = list(ex.map(_compile, SOURCES))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print("built", LIB)
    return LIB


if __name__ == "__main__":
    build()
