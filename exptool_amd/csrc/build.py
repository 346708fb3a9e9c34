"""Build libexptool_bfe.so (gfx950) from the HIP sources in this directory.

    python -m exptool_amd.csrc.build [-j N] [--clean]

Each .hip file is compiled with hipcc to an object under exptool_amd/_build/
and the objects are linked into exptool_amd/libexptool_bfe.so (in-tree, so it
travels with the source tree).  Packed-FP32 instruction selection is disabled
(-packed-fp32-ops) on every device compile.
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.dirname(HERE)
BUILD = os.path.join(PKG, "_build")
LIB = os.path.join(PKG, "libexptool_bfe.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("BFE_OFFLOAD_ARCH", "gfx950")

CXXFLAGS = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-result",
]
# The step loops of the orbit kernels: machine LICM moves the constants of the
# inlined field evaluation (logarithm series, reciprocals) into registers that
# stay live over the whole loop, which spills them; materialised where they are
# used they cost a scalar move each (leapfrog kernel 316-340 B spilled per lane
# -> 0; 1M orbits 76.2 -> 70.3 us a step, RK4 105 -> 99 us an evaluation, same
# results).
EXTRA = {"bfe_leapfrog.hip": ["-mllvm", "-disable-machine-licm"]}


def sources():
    return sorted(f for f in os.listdir(HERE) if f.endswith(".hip"))


def compile_one(src):
    obj = os.path.join(BUILD, src[:-4] + ".o")
    cmd = [HIPCC, *CXXFLAGS, *EXTRA.get(src, []), "-c", os.path.join(HERE, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stdout}\n{r.stderr}")
    return obj, r.stderr


def build(jobs=None, verbose=False):
    os.makedirs(BUILD, exist_ok=True)
    srcs = sources()
    jobs = jobs or min(len(srcs), os.cpu_count() or 4, 8)
    objs = []
    with cf.ThreadPoolExecutor(jobs) as ex:
        for obj, err in ex.map(compile_one, srcs):
            objs.append(obj)
            if verbose and err.strip():
                print(err, file=sys.stderr)
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "-shared", f"--offload-arch={ARCH}", "-o", tmp, *objs,
           "-Wl,-rpath,/opt/rocm/lib"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("-j", type=int, default=None)
    ap.add_argument("--clean", action="store_true")
    ap.add_argument("-v", action="store_true")
    a = ap.parse_args()
    if a.clean and os.path.isdir(BUILD):
        shutil.rmtree(BUILD)
    print(build(a.j, a.v))
