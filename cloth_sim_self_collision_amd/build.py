"""Builds the HIP library libclothsim.so in-tree for gfx950.

    python -m cloth_sim_self_collision_amd.build

Every translation unit is compiled with hipcc; device code uses
-ffp-contract=off (no fused multiply-add contraction: each double operation
rounds once, in source order, like the reference's x86-64 build) and
packed FP32 disabled.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "libclothsim.so")
BUILD_DIR = os.path.join(HERE, "_build")

SOURCES = ["cs_setup.cpp", "cs_setup_cache.cpp", "cs_strips.cpp", "cs_api.cpp", "cs_solve.hip",
           "cs_strips.hip", "cs_contact.hip",
           "cs_elements.hip", "cs_noalloc.hip"]
HEADERS = ["cs_math.hpp", "cs_ordered_sum.hpp", "cs_item_sum.hpp",
           "cs_setup.hpp", "cs_strips.hpp",
           "cs_device.hpp", "cs_solve.hpp", "cs_contact.hpp"]

ARCH = os.environ.get("CLOTHSIM_ARCH", "gfx950")
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
    "-fno-fast-math", "-Wall", "-Wno-unused-function", "-Wno-unused-result",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", os.path.join(ROOT, "include"),
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found")


def _compile(src: str) -> str:
    obj = os.path.join(BUILD_DIR, src + ".o")  # cs_strips.cpp and cs_strips.hip differ
    cmd = [hipcc()] + FLAGS + ["-c", os.path.join(CSRC, src), "-o", obj]
    if src.endswith(".cpp"):
        cmd[1:1] = ["-x", "hip"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed: {src}\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    warn = (r.stdout + r.stderr).strip()
    if warn:
        lines = [ln for ln in warn.splitlines() if "packed-fp32-ops" not in ln and ln.strip()]
        if lines:
            sys.stderr.write("\n".join(lines) + "\n")
    return obj


def build(jobs: int = 8) -> str:
    """Compile all sources and link libclothsim.so; returns its path."""
    os.makedirs(BUILD_DIR, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=max(1, min(jobs, len(SOURCES)))) as ex:
        objs = list(ex.map(_compile, SOURCES))
    tmp = OUT + ".tmp"
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, OUT)
    return OUT


if __name__ == "__main__":
    print(build())
