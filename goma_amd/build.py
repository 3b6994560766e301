"""Builds libgm.so (HIP for gfx950 + host C++) in-tree with hipcc.

Every source is compiled on each call; the shared library lands next to this
file as goma_amd/libgm.so.
"""
from __future__ import annotations

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libgm.so")
OBJ = os.path.join(HERE, "_build")

SOURCES = ["gm_setup.cpp", "gm_capi.cpp", "gm_hier.cpp", "gm_fill.hip", "gm_gather.hip", "gm_linalg.hip", "gm_mg.hip", "gm_mlp.hip",
           "gm_band.hip"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
# packed-FP32 instructions are disabled for device code (they have given
# silently wrong results on this hardware); the host pass warns it does not
# know the feature, which is harmless.
DEVICE_FLAGS = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
COMMON = ["-O3", "-fPIC", "-std=c++17", "-fopenmp", f"--offload-arch={ARCH}", "-Wall",
          "-Wno-unused-function", "-Wno-unused-variable", "-Wno-unused-result", "-Wno-unused-value"]


def _run(cmd):
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("build failed: " + " ".join(cmd))
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l and l.strip())
    return err


def build(verbose: bool = False) -> str:
    os.makedirs(OBJ, exist_ok=True)
    objs = []
    for s in SOURCES:
        src = os.path.join(CSRC, s)
        obj = os.path.join(OBJ, s + ".o")
        cmd = [HIPCC] + COMMON + DEVICE_FLAGS + ["-c", src, "-o", obj]
        if s.endswith(".hip"):
            cmd[1:1] = ["-x", "hip"]
        msg = _run(cmd)
        if verbose and msg:
            print(msg)
        objs.append(obj)
    tmp = LIB + ".tmp"
    _run([HIPCC, "-shared", "-fopenmp", f"--offload-arch={ARCH}", "-o", tmp] + objs)
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
