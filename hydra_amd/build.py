"""Builds libhydra_hip.so in-tree for gfx950 with hipcc.

    python -m hydra_amd.build [--jobs N]

Each .hip source is compiled to an object in hydra_amd/_build/, then linked into
hydra_amd/libhydra_hip.so. Always recompiles (this is also the CPU-side "does it build" check).
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import shutil
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libhydra_hip.so")
SOURCES = ["hh_api.hip", "hh_route.hip", "hh_gemm.hip", "hh_gemm_block.hip", "hh_prefill.hip", "hh_ops.hip", "hh_attn.hip", "hh_block.hip", "hh_proj.hip"]


def hipcc() -> str:
    for cand in [os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")]:
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (ROCm is required to build HydraHIP)")


FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # No fused multiply-add contraction beyond the explicit fmaf calls: the arithmetic of every
    # output element is then fixed by the source, identical in decode and prefill.
    "-ffp-contract=off",
    # Packed fp32 instructions stay off.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-variable", "-Wno-unused-but-set-variable",
]


DEFINES: list = []   # extra -D flags (development variants, e.g. HH_TRACE); none by default


def compile_one(src: str) -> str:
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    cmd = [hipcc(), *FLAGS, *[f"-D{d}" for d in DEFINES], "-I", os.path.join(ROOT, "include"), "-I", CSRC, "-c",
           os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{r.stdout}\n{r.stderr}")
    return obj


def build(jobs: int = 4) -> str:
    os.makedirs(BUILD, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=max(1, jobs)) as ex:
        objs = list(ex.map(compile_one, SOURCES))
    tmp = LIB + ".tmp"
    r = subprocess.run([hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs],
                       capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=4)
    ap.add_argument("--define", action="append", default=[],
                    help="extra preprocessor definition (development variants)")
    args = ap.parse_args()
    DEFINES.extend(args.define)
    print(build(args.jobs))
