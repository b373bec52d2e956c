"""Builds librsh_scatter.so in-tree with hipcc for gfx950.

Every HIP translation unit under csrc/ is compiled in parallel; host-only C++
units are compiled by hipcc as host code. The shared library lands next to
this file, where relativistic_solver_hllc_amd._native loads it from.

Usage:  python -m relativistic_solver_hllc_amd.build   (or build() from Python)
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
REPO_DIR = os.path.dirname(PKG_DIR)
CSRC = os.path.join(PKG_DIR, "csrc")
OBJ_DIR = os.path.join(PKG_DIR, "_build")
LIB_NAME = "librsh_scatter.so"
LIB_PATH = os.path.join(PKG_DIR, LIB_NAME)

ARCH = os.environ.get("RSH_OFFLOAD_ARCH", "gfx950")
HIPCC = os.environ.get("HIPCC", shutil.which("hipcc") or "/opt/rocm/bin/hipcc")

# Packed-FP32 instructions are disabled for all device code (v_pk_*_f32 forms
# have produced silently wrong results on these machines).
DEVICE_FLAGS = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
COMMON = ["-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function", f"-I{REPO_DIR}/include", f"-I{CSRC}"]

HIP_SOURCES = ["kernels_f64.hip", "kernels_f64_reg.hip", "kernels_split.hip", "kernels_iter.hip", "kernels_iter_split.hip",
               "kernels_moments.hip", "kernels_split_resident.hip", "kernels_sweep.hip", "kernels_peak.hip", "noalloc.hip"]
# Resident-panel split kernels, grouped iteration and single problem: an unrolled instance per K-step count and form,
# in twelve units that compile in parallel.
RES_SOURCES = [f"kernels_{kind}_{form}_{part}.hip" for kind in ("iter_res", "res")
               for form in ("bf16x2", "fp16x2", "bf16x3") for part in "ab"]
HIP_SOURCES = ["kernels_split_resident.hip", *RES_SOURCES,
               *(s for s in HIP_SOURCES if s != "kernels_split_resident.hip")]  # longest first
HOST_SOURCES = ["capi.cpp", "batch.cpp", "server.cpp", "sweep.cpp", "sweep_prep.cpp"]
# Per-source device flags. The resident-panel split kernels add each K-step's
# fresh FP32 products to its main sums with VALU adds: with MFMA results in
# VGPRs (instead of AGPRs read back one register at a time) it ran 3-8 % faster.
EXTRA_FLAGS = {s: ["-mllvm", "-amdgpu-mfma-vgpr-form"] for s in ["kernels_split_resident.hip", *RES_SOURCES]}

# Drop-in shim of the reference's cuda_solve.h names (stand-alone types) and the
# test driver that replays the reference's call sequence through it.
SHIM_SRC = os.path.join(PKG_DIR, "shim", "cuda_solve_shim.cpp")
SHIM_DRIVER_SRC = os.path.join(REPO_DIR, "tests", "shim", "shim_driver.cpp")
SHIM_DRIVER = os.path.join(OBJ_DIR, "shim_driver")


def _run(cmd):
    proc = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass warns that it does not know the packed-fp32 feature; drop that noise
    err = "\n".join(l for l in proc.stderr.splitlines() if "packed-fp32-ops" not in l)
    if proc.returncode != 0:
        raise RuntimeError(f"command failed ({proc.returncode}): {' '.join(cmd)}\n{err}")
    return err


def _compile(src: str) -> str:
    path = os.path.join(CSRC, src)
    obj = os.path.join(OBJ_DIR, os.path.splitext(src)[0] + ".o")
    if src.endswith(".hip"):
        cmd = [HIPCC, f"--offload-arch={ARCH}", *COMMON, *DEVICE_FLAGS, *EXTRA_FLAGS.get(src, []), "-x", "hip", "-c",
               path, "-o", obj]
    else:
        cmd = [HIPCC, *COMMON, "-c", path, "-o", obj]
    _run(cmd)
    return obj


def build(verbose: bool = False) -> str:
    """Compiles every source and links LIB_PATH; returns the library path."""
    os.makedirs(OBJ_DIR, exist_ok=True)
    sources = HIP_SOURCES + HOST_SOURCES
    workers = min(len(sources), max(1, min(8, os.cpu_count() or 1)))
    with ThreadPoolExecutor(max_workers=workers) as ex:
        objs = list(ex.map(_compile, sources))
    tmp = LIB_PATH + ".tmp"
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp])
    os.replace(tmp, LIB_PATH)
    _run(["g++", "-std=c++17", "-O2", "-Wall", f"-I{REPO_DIR}/include", SHIM_SRC, SHIM_DRIVER_SRC,
          f"-L{PKG_DIR}", "-lrsh_scatter", f"-Wl,-rpath,{PKG_DIR}", "-Wl,-rpath,$ORIGIN/..", "-o", SHIM_DRIVER])
    if verbose:
        print("built", LIB_PATH, "and", SHIM_DRIVER)
    return LIB_PATH


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
