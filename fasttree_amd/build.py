"""Builds libfasttree_amd.so (gfx950) from fasttree_amd/csrc/*.hip with hipcc.

Usage: python -m fasttree_amd.build [--jobs N]
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import glob
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libfasttree_amd.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("FT_OFFLOAD_ARCH", "gfx950")

# -ffp-contract=off: the FP64 squared distance is (dx*dx + dy*dy) + dz*dz with
# every product and sum rounded, never fused.  Packed FP32 instructions are
# disabled for all device code.
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-fPIC", "-std=c++17", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-result",
]

# The traversal sources only: -structurizecfg-skip-uniform-regions.  LLVM's CFG
# structurizer then leaves regions whose branches are all wave-uniform (wave
# votes, loop exits on a ballot) as they are; divergent regions are structurized
# as before.  Structurized, the traversal's insertion loop (uniform branches
# only) gets flow blocks that merge all 32 register-resident top-k keys, and the
# register allocator then keeps the list in two register sets and copies it
# between them every round (about 980 v_mov_b64 in the self-kNN kernel of 10M
# 64-bit points, 143 without; 168 -> 142 VGPRs; the kernel 23.7 -> 21.2 ms).
#
# What it breaks, and these sources therefore avoid: a lane flag (a bool kept as
# a mask of the wave) that has a value on the way around a divergent branch and
# gets another inside it, behind a wave-uniform branch:
#     bool left = tied;                    // per lane
#     if (!left) left = store_row(...);    // divergent; uniform branches inside
# At the join the mask of the lanes inside replaces the whole mask (seen in the
# assembly: `s_or_b64 left, a, b` where the structurized code has
# `s_orn2_b64 left, bad, exec`), so lanes that went around lose their bit.
# Flags of that kind are wave masks voted outside divergent branches
# (__ballot), or counts in a vector register.
TRAVERSAL = {"ft_query.hip", "ft_batch.hip"}
TRAVERSAL_FLAGS = ["-mllvm", "-structurizecfg-skip-uniform-regions"]


def _compile(src: str) -> str:
    obj = os.path.join(OBJ, os.path.basename(src) + ".o")
    extra = TRAVERSAL_FLAGS if os.path.basename(src) in TRAVERSAL else []
    cmd = [HIPCC, *FLAGS, *extra, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr[-6000:]}")
    return obj


def build(jobs: int = 4, verbose: bool = True) -> str:
    os.makedirs(OBJ, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    with cf.ThreadPoolExecutor(max_workers=max(1, jobs)) as ex:
        objs = list(ex.map(_compile, srcs))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr[-6000:]}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=4)
    a = ap.parse_args()
    try:
        build(a.jobs)
    except RuntimeError as e:
        print(e, file=sys.stderr)
        sys.exit(1)
