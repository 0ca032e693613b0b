"""Builds libohpic.so (gfx950 HIP kernels + C ABI) in-tree with hipcc.

Usage: ``python -m ohhelppic3d_amd.build`` or ``ohhelppic3d_amd.build.build()``.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
OBJ = os.path.join(PKG, "_build")
LIB = os.path.join(PKG, "libohpic.so")

SOURCES = ["ohpic_particles.hip", "ohpic_particles_mixed.hip", "ohpic_fields.hip",
           "ohpic_fft.hip", "ohpic_ops.hip", "ohpic_api.cpp", "ohpic_snapshot.cpp"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("OHPIC_ARCH", "gfx950")

# -packed-fp32-ops keeps the compiler from emitting packed FP32 VALU ops.
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-fPIC", "-std=c++17", "-Wall",
    "-Wno-unused-result", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I" + os.path.join(ROOT, "include"),
]

# The particle kernels without the atomic optimizer: it turns one lane's LDS
# counter add into a wave-wide reduction that waits for its result at once,
# while they need it only after the charge deposit.  Their counters that many
# lanes add to are combined in the source (count_lanes, wave_counter_add).
SOURCE_FLAGS = {src: ["-mllvm", "-amdgpu-atomic-optimizer-strategy=None"]
                for src in ("ohpic_particles.hip", "ohpic_particles_mixed.hip")}


def _compile(src: str) -> str:
    out = os.path.join(OBJ, os.path.splitext(src)[0] + ".o")
    lang = ["-x", "hip"]
    cmd = [HIPCC, *FLAGS, *SOURCE_FLAGS.get(src, []), *lang, "-c", os.path.join(CSRC, src), "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr[-6000:]}")
    return out


def build(verbose: bool = False) -> str:
    """Compile every source for gfx950 and link libohpic.so; returns its path."""
    os.makedirs(OBJ, exist_ok=True)
    with ThreadPoolExecutor(max_workers=min(6, len(SOURCES))) as ex:
        objs = list(ex.map(_compile, SOURCES))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs, "-ldl"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr[-6000:]}")
    os.replace(tmp, LIB)
    if verbose:
        print("built", LIB)
    return LIB


def clean() -> None:
    shutil.rmtree(OBJ, ignore_errors=True)
    if os.path.exists(LIB):
        os.remove(LIB)


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
