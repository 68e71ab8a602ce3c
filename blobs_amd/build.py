"""Build the in-tree native libraries.

* ``blobs_amd/libblobs_gpu.so``   -- HIP kernels for gfx950 + the C ABI of
  include/blobs_gpu.h (hipcc, one object per source, compiled in parallel).
* ``blobs_amd/libblobs_scenes.so`` -- synthetic scene generator (plain C).

Every HIP source is compiled with ``-ffp-contract=off`` (bit-exact parity
with the reference's un-fused f32 arithmetic) and with packed-FP32 code
generation disabled.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
BUILD = PKG / "_build"
ROOT = PKG.parent

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("BLOBS_OFFLOAD_ARCH", "gfx950")

HIP_SOURCES = ["sort.hip", "step_kernels.hip", "sphere_kernels.hip", "export_kernels.hip", "ordered_contacts.hip", "spatial.hip", "diff_kernels.hip", "batch_kernels.hip", "small_kernels.hip", "world.cpp", "batch.cpp",
               "diff.cpp", "capi.cpp"]
HIP_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-fno-fast-math",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
    "-Wno-unused-variable",
    "-Wno-unused-lambda-capture",
    "-I", str(ROOT / "include"),
]


def _run(cmd: list[str]) -> None:
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(" ".join(cmd) + "\n" + r.stdout + r.stderr)
        raise RuntimeError(f"command failed ({r.returncode}): {cmd[0]} ... {cmd[-1]}")
    # surface warnings other than the known host-pass note about packed-fp32-ops
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l and l.strip())
    if err.strip():
        sys.stderr.write(err + "\n")


def _compile(src: str) -> Path:
    out = BUILD / (src.replace(".", "_") + ".o")
    _run([HIPCC, *HIP_FLAGS, "-x", "hip", "-c", str(CSRC / src), "-o", str(out)])
    return out


def build_gpu(jobs: int | None = None) -> Path:
    BUILD.mkdir(exist_ok=True)
    sources = [s for s in HIP_SOURCES if (CSRC / s).exists()]
    jobs = jobs or min(len(sources), max(1, (os.cpu_count() or 2)))
    with cf.ThreadPoolExecutor(jobs) as ex:
        objs = list(ex.map(_compile, sources))
    lib = PKG / "libblobs_gpu.so"
    tmp = PKG / "libblobs_gpu.so.tmp"
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)])
    os.replace(tmp, lib)
    return lib


def build_scenes() -> Path:
    lib = PKG / "libblobs_scenes.so"
    tmp = PKG / "libblobs_scenes.so.tmp"
    _run(["gcc", "-O2", "-std=c11", "-fPIC", "-shared", "-ffp-contract=off", "-Wall", "-Wextra",
          "-o", str(tmp), str(CSRC / "scenegen.c"), "-lm"])
    os.replace(tmp, lib)
    return lib


def build_all() -> None:
    build_scenes()
    build_gpu()


if __name__ == "__main__":
    build_all()
    print("built", PKG / "libblobs_gpu.so", PKG / "libblobs_scenes.so")
