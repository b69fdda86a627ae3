"""Builds the engine library triplelens_amd/lib/liblcirs.so with hipcc for gfx950.

All code (host and device) is compiled with -ffp-contract=off: the ray test
and the seed search must round exactly as the IEEE operations are written.
Packed FP32 instructions are disabled (-packed-fp32-ops); the engine's hot
paths are FP64 anyway.
"""
from __future__ import annotations

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIBDIR, "liblcirs.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SOURCES = ["tl_kernels.hip", "tl_api.cpp", "tl_mlp.hip", "tl_surrogate.cpp"]
FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    "-ffp-contract=off",
    "-fno-fast-math",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # host functions on cache lines of their own: the network's initial weights
    # (200,000 normal draws) took 8 or 14 ms, depending on where they fell
    "-falign-functions=64",
    "-Wall",
    "-Wno-unused-function",
]


def build(verbose: bool = False) -> str:
    os.makedirs(LIBDIR, exist_ok=True)
    tmp = LIB + ".tmp"
    cmd = [HIPCC] + FLAGS + [os.path.join(CSRC, s) for s in SOURCES] + ["-o", tmp]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        sys.stderr.write(res.stdout + res.stderr)
        raise RuntimeError("hipcc failed to build liblcirs.so")
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
