"""Build the HIP library libplasmasim.so for gfx950 with hipcc, in-tree.

Each translation unit is compiled to an object with its own floating-point
contraction setting: the FP64 plain form must round every operation as the
reference's C does (-ffp-contract=off); the FP32 form may fuse.  Packed FP32
instructions are disabled for all device code.
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "libplasmasim.so")
BUILD = os.path.join(HERE, "_build")

ARCH = os.environ.get("PIC_OFFLOAD_ARCH", "gfx950")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

COMMON = [
    "-O3", "-fPIC", "-std=c++17", f"--offload-arch={ARCH}",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-munsafe-fp-atomics", "-Wall", "-Wno-unused-function",
    "-Wno-unused-variable", "-Wno-unused-parameter",
]
UNITS = {
    "pic_api.hip": ["-ffp-contract=off"],
    "pic_fp64.hip": ["-ffp-contract=off"],
    # fused by expression (on), not by what the optimiser finds (fast): every
    # instantiation of the particle pass rounds alike, at the same number of
    # instructions.  The pass schedules better with memory clauses kept
    # together (1.2 % faster pass at 128^3 x 64 ppc)
    "pic_fp32.hip": ["-ffp-contract=on", "-mllvm", "-amdgpu-sched-strategy=max-memory-clause"],
    "pic_prim.hip": ["-ffp-contract=off"],
    "pic_adj.hip": ["-ffp-contract=off"],
    "pic2d_api.hip": ["-ffp-contract=off"],
    "pic2d_fields.hip": ["-ffp-contract=off"],
    "pic2d_particles.hip": ["-ffp-contract=off"],
    "pic_ckpt.hip": ["-ffp-contract=off"],
    "pic_output.cpp": ["-ffp-contract=off"],
    "pic_poisson.hip": ["-ffp-contract=off"],
    "pic_noalloc.hip": ["-ffp-contract=off"],
}


def _compile(src, flags):
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC] + COMMON + flags + ["-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stdout}\n{r.stderr}")
    return obj


def build(verbose=True):
    os.makedirs(BUILD, exist_ok=True)
    with ThreadPoolExecutor(max_workers=8) as ex:
        objs = list(ex.map(lambda kv: _compile(*kv), UNITS.items()))
    tmp = OUT + ".tmp"
    cmd = [HIPCC, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, OUT)
    # the C host driver (fdtd()/main_func() restated over the C-ABI)
    drv = os.path.join(HERE, "driver")
    cmd = ["gcc", "-O2", "-std=gnu11", "-Wall", "-o", os.path.join(drv, "pic_run"),
           os.path.join(drv, "pic_run.c"), "-L" + HERE, "-lplasmasim",
           "-Wl,-rpath,$ORIGIN/.."]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"driver build failed:\n{r.stdout}\n{r.stderr}")
    if verbose:
        print(f"built {OUT} and driver/pic_run")
    return OUT


if __name__ == "__main__":
    build()
    sys.exit(0)
