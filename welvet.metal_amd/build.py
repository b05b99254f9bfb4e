"""Builds libwelvet_hip.so (HIP kernels + C ABI) for gfx950, in-tree, and the
wire tool welvet_dense_fwd (host C++ over the C ABI, linked to that library).

    python welvet.metal_amd/build.py            # build
    python welvet.metal_amd/build.py --jobs 8   # parallel object compiles

Every object is rebuilt on each call.  Flags:
  -ffp-contract=off     codec arithmetic must round each step (q*s + min never
                        fuses); kernels that want FMA call fma/fmaf explicitly
  -packed-fp32-ops off  no packed fp32 add / mul / fma instructions: some of
                        their forms have given sporadic wrong results on
                        MI355X machines without raising an error
  -fvisibility=hidden   only the welvet_c.h entry points are exported
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libwelvet_hip.so")
TOOL = os.path.join(HERE, "welvet_dense_fwd")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")
CXX = os.environ.get("CXX", "g++")
SOURCES = ["codec.hip", "dense.hip", "runtime.cpp", "volume.cpp", "swiglu.cpp", "chain.cpp", "model.cpp"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

FLAGS = [
    "-O3", "-std=c++17", "-fPIC", "--offload-arch=gfx950", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-fvisibility=hidden", "-Wall", "-Wno-unused-function", "-Wno-unused-variable",
    "-Wno-unknown-pragmas",
]


def _compile(src: str) -> tuple[str, str]:
    obj = os.path.join(BUILD, src + ".o")
    cmd = [HIPCC, *FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    if src.endswith(".cpp"):
        cmd[1:1] = ["-x", "hip"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed: {src}\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    return obj, r.stderr


def build(jobs: int = 3, verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=max(1, jobs)) as ex:
        results = list(ex.map(_compile, SOURCES))
    if verbose:
        for _, err in results:
            if err.strip():
                print(err, file=sys.stderr)
    objs = [o for o, _ in results]
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    build_tool()
    return LIB


def build_tool() -> str:
    """The wire tool: host code only, finds the library next to itself."""
    tmp = TOOL + ".tmp"
    cmd = [CXX, "-O2", "-std=c++17", "-Wall", "-I", INCLUDE, os.path.join(CSRC, "wire_tool.cpp"),
           "-o", tmp, "-L", HERE, "-lwelvet_hip", "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"tool build failed\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, TOOL)
    return TOOL


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=3)
    ap.add_argument("-v", "--verbose", action="store_true")
    a = ap.parse_args()
    print(build(a.jobs, a.verbose))
