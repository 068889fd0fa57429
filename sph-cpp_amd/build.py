"""Build recipe for libpbf.so (hipcc, gfx950) and the C++ host driver.

Run ``python sph-cpp_amd/build.py`` or call :func:`build`.  Everything is
built in-tree: ``sph-cpp_amd/libpbf.so`` and ``sph-cpp_amd/sph_run``.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
HOST = os.path.join(HERE, "host")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libpbf.so")
RUNNER = os.path.join(HERE, "sph_run")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SOURCES = ["pbf_api.hip", "pbf_grid.hip", "pbf_passes.hip", "pbf_fused.hip", "pbf_mlp.hip", "pbf_check.hip",
           "pbf_noalloc.hip", "pbf_transfer.hip"]

# -ffp-contract=off: no fused multiply-add, every op rounds like the reference.
# HIP's default single-precision divide and sqrt are correctly rounded; the
# flag is spelled out so that a changed default cannot slip in.
# Packed FP32 instructions are disabled.
HIP_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
    "-Wno-unused-value",
    "-I" + os.path.join(ROOT, "include"),
]


def _run(cmd: list[str]) -> None:
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in res.stdout.splitlines() if "packed-fp32-ops" not in l)
    if res.returncode != 0:
        raise RuntimeError("build failed: " + " ".join(cmd) + "\n" + out)
    if out.strip():
        sys.stderr.write(out + "\n")


def build(verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    objs = []
    cmds = []
    for src in SOURCES:
        obj = os.path.join(BUILD, src.replace(".hip", ".o"))
        objs.append(obj)
        cmds.append([HIPCC, *HIP_FLAGS, "-c", os.path.join(CSRC, src), "-o", obj])
    with ThreadPoolExecutor(max_workers=len(cmds)) as ex:
        list(ex.map(_run, cmds))
    tmp = LIB + ".tmp"
    _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-Wl,--no-undefined", "-o", tmp, *objs,
          "-L/opt/rocm/lib", "-lrocprofiler-sdk-roctx", "-Wl,-rpath,/opt/rocm/lib"])
    os.replace(tmp, LIB)
    # C++ host driver over the C ABI (restates Simulation/Source/main.cpp)
    drv = os.path.join(HOST, "sph_main.cpp")
    if os.path.exists(drv):
        _run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I" + os.path.join(ROOT, "include"),
              "-I" + HOST, drv, "-o", RUNNER, "-L" + HERE, "-lpbf", "-Wl,-rpath,$ORIGIN"])
    if verbose:
        print("built", LIB)
    return LIB


if __name__ == "__main__":
    build(verbose=True)
