"""Build recipes for the native parts of lvr2_amd.

- liblvrhip.so   : the gfx950 HIP library behind include/lvrhip.h (hipcc)
- libscenes.so   : the seeded synthetic scene generators (g++/OpenMP, host only)

Run ``python -m lvr2_amd.build`` or call :func:`build_all`.
"""
from __future__ import annotations

import os
import shlex
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(ROOT, "include")

LIB = os.path.join(HERE, "liblvrhip.so")
SCENES = os.path.join(HERE, "libscenes.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

# -ffp-contract=off: the kNN key d^2 and the ordered fp32 sums must round as written.
# Packed fp32 ops are disabled for all device code.
HIP_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
]


def _run(cmd: list[str]) -> None:
    print("+", " ".join(shlex.quote(c) for c in cmd), flush=True)
    subprocess.run(cmd, check=True)


# The library's translation units, compiled in parallel and linked into one shared object.
HIP_UNITS = ["lvrhip", "knn_tile_p8", "knn_tile_p4", "knn_tile_p2"]


def build_lib() -> str:
    with tempfile.TemporaryDirectory(prefix="lvrhip_build_") as tmpdir:
        objs = [os.path.join(tmpdir, u + ".o") for u in HIP_UNITS]
        procs = []
        for u, o in zip(HIP_UNITS, objs):
            cmd = [HIPCC, *HIP_FLAGS, f"-I{INCLUDE}", f"-I{CSRC}", "-c", os.path.join(CSRC, u + ".hip"), "-o", o]
            print("+", " ".join(shlex.quote(c) for c in cmd), flush=True)
            procs.append((cmd, subprocess.Popen(cmd)))
        failed = [(cmd, p.returncode) for cmd, p in procs if p.wait() != 0]
        if failed:
            raise subprocess.CalledProcessError(failed[0][1], failed[0][0])
        tmp = LIB + ".tmp"
        _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp])
        os.replace(tmp, LIB)
    return LIB


def build_scenes() -> str:
    src = os.path.join(CSRC, "scenes.cpp")
    tmp = SCENES + ".tmp"
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fopenmp", src, "-o", tmp])
    os.replace(tmp, SCENES)
    return SCENES


def build_all() -> None:
    build_scenes()
    build_lib()


if __name__ == "__main__":
    what = sys.argv[1:] or ["all"]
    for w in what:
        {"all": build_all, "lib": build_lib, "scenes": build_scenes}[w]()
