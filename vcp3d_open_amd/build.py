"""Builds the in-tree gfx950 libraries with hipcc: vcp3d_open_amd/libvcp3d_amd.so
(the path) and vcp3d_open_amd/libvcp3d_ab.so (the VALU / MFMA interpolation
measurement that bench.py --workload interpolation runs)."""
from __future__ import annotations

import concurrent.futures
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
ROOT = os.path.dirname(HERE)
LIB = os.path.join(HERE, "libvcp3d_amd.so")
AB_LIB = os.path.join(HERE, "libvcp3d_ab.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SOURCES = ["kernels.hip", "geometry.hip", "setup.cpp", "capi.cpp", "batch.cpp", "contraction_ab.hip"]
AB_SOURCES = ["contraction_ab.hip"]
# compiled once per shape (nDOFs1D, nInt1D)
SHAPE_SOURCES = ["volume.hip", "volume_workgroup.hip", "face.hip"]
SHAPES = [(3, 4), (4, 5), (4, 6), (5, 7), (6, 8), (7, 9)]
# per-source flags: the device metric terms repeat the host set-up's
# arithmetic exactly, so neither side contracts multiply-adds
EXTRA = {"geometry.hip": ["-ffp-contract=off"], "setup.cpp": ["-ffp-contract=off"]}
COMMON = ["-O3", "-fPIC", "-std=c++17", "--offload-arch=gfx950",
          # no packed FP32 instructions anywhere in device code
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
          "-I" + CSRC, "-I" + os.path.join(ROOT, "include")]


def build(verbose: bool = False) -> str:
    objdir = os.path.join(HERE, "_build")
    os.makedirs(objdir, exist_ok=True)
    units = [(src, os.path.splitext(src)[0] + ".o", EXTRA.get(src, [])) for src in SOURCES]
    units += [(src, f"{os.path.splitext(src)[0]}_{k}_{m}.o", [f"-DVCP_SHAPE_K={k}", f"-DVCP_SHAPE_M={m}"])
              for src in SHAPE_SOURCES for k, m in SHAPES]

    def compile_unit(unit):
        src, obj, flags = unit
        cmd = [HIPCC, *COMMON, *flags, "-x", "hip", "-c", os.path.join(CSRC, src), "-o", os.path.join(objdir, obj)]
        if verbose:
            print(" ".join(cmd), flush=True)
        return subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)

    failed = []
    jobs = min(8, os.cpu_count() or 1)
    with concurrent.futures.ThreadPoolExecutor(jobs) as pool:
        for (src, obj, _), p in zip(units, pool.map(compile_unit, units)):
            if p.returncode != 0:
                failed.append(obj)
                sys.stderr.write(p.stdout)
            elif verbose and p.stdout.strip():
                sys.stderr.write(p.stdout)
    if failed:
        raise RuntimeError("hipcc failed for " + ", ".join(failed))
    for lib, ab in ((LIB, False), (AB_LIB, True)):
        tmp = lib + ".tmp"
        objs_l = [os.path.join(objdir, obj) for src, obj, _ in units if (src in AB_SOURCES) == ab]
        cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs_l]
        subprocess.run(cmd, check=True)
        os.replace(tmp, lib)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
