"""Build the HIP library in-tree with hipcc for gfx950.

    python -m gms_liberi_amd.build            # -> gms_liberi_amd/libliberi_hip.so

The kernels of the 55 integral classes are spread over translation units of
about equal compile time, which compile in parallel; the host orchestration is
one more unit.  Every HIP unit is compiled with packed FP32 disabled
(`-target-feature -packed-fp32-ops`).
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

from .census import CLASS_L

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
OBJ = PKG / "_build"
LIB = PKG / "libliberi_hip.so"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

COMMON = ["--offload-arch=" + ARCH, "-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function",
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", str(PKG.parent / "include")]


# units the class kernels are spread over (each carries its own copy of the Rys tables)
KERNEL_UNITS = 16
# launches shared by several small classes, a unit each
SHARED_LAUNCHES = 6
# seconds a class's kernels take to compile, where that is above 5 (the wave-split forms)
COMPILE_S = {36: 97, 38: 87, 19: 39, 35: 35, 37: 15, 33: 15, 30: 15, 14: 14, 15: 12, 29: 11, 18: 10, 34: 10, 17: 6}


def kernel_units() -> list:
    """Class ids of each unit, the longest compile first onto the unit with the least so far."""
    cost = {c: COMPILE_S.get(c, 4) for c in range(len(CLASS_L))}
    units = [[] for _ in range(KERNEL_UNITS)]
    for c in sorted(cost, key=cost.get, reverse=True):
        min(units, key=lambda u: sum(cost[x] for x in u)).append(c)
    return units


def _run(cmd):
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(" ".join(cmd) + "\n" + r.stdout + r.stderr)
        raise RuntimeError(f"compile failed: {cmd[-1]}")
    return r


def build(verbose: bool = True) -> Path:
    OBJ.mkdir(exist_ok=True)
    kernels = [HIPCC, *COMMON, "-c", str(CSRC / "eri_kernels.hip")]
    jobs = [[*kernels, "-DLIBERI_UNIT=-3", "-o", str(OBJ / "eri_fused.o")]]
    for k in range(SHARED_LAUNCHES):
        jobs.append([*kernels, f"-DLIBERI_UNIT={-10 - k}", "-o", str(OBJ / f"eri_shared{k}.o")])
    for g, classes in enumerate(kernel_units()):
        entries = " ".join("X(%d, %d, %d, %d, %d)" % (c, *CLASS_L[c]) for c in classes)
        jobs.append([*kernels, "-DLIBERI_UNIT=1", f"-DLIBERI_UNIT_LIST(X)={entries}", "-o", str(OBJ / f"eri_g{g}.o")])
    jobs.append([*kernels, "-DLIBERI_UNIT=-1", "-o", str(OBJ / "eri_common.o")])
    jobs.append([HIPCC, *COMMON, "-c", str(CSRC / "api.cpp"), "-o", str(OBJ / "api.o")])
    jobs.append([HIPCC, *COMMON, "-c", str(CSRC / "noalloc.hip"), "-o", str(OBJ / "noalloc.o")])
    nproc = min(len(jobs), int(os.environ.get("MAX_JOBS", os.cpu_count() or 4)))
    with ThreadPoolExecutor(nproc) as ex:
        list(ex.map(_run, jobs))
    objs = [j[-1] for j in jobs]
    tmp = LIB.with_suffix(".so.tmp")
    _run([HIPCC, "--offload-arch=" + ARCH, "-shared", "-fPIC", "-o", str(tmp), *objs])
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build()
