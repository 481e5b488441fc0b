"""Builds libopengenie_amd.so (gfx950) and its CPython binding _native from
opengenie_amd/csrc with hipcc.

Usage: python -m opengenie_amd.build [--jobs N]

Every .hip source is compiled to an object in parallel, then linked into one
shared library next to this file; pycall.cpp (host code) becomes the module
_native of this interpreter beside it, linked to the library (without the
interpreter's headers there is none, and the wrappers call through ctypes).
Flags of the device sources:
  --offload-arch=gfx950         CDNA4 (MI355X) only
  -ffp-contract=off             no silent a*b+c fusion (bit-exact rounding)
  -target-feature -packed-fp32-ops
                                no v_pk_{add,mul,fma}_f32 generation
"""

from __future__ import annotations

import argparse
import glob
import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_NAME = "libopengenie_amd.so"
LIB_PATH = os.path.join(HERE, LIB_NAME)
NATIVE_PATH = os.path.join(HERE, "_native" + sysconfig.get_config_var("EXT_SUFFIX"))
BUILD_DIR = os.path.join(HERE, "_build")

ARCH = "gfx950"
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (ROCm is required to build opengenie_amd)")


def sources() -> list[str]:
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(src: str) -> str:
    obj = os.path.join(BUILD_DIR, os.path.basename(src)[:-4] + ".o")
    cmd = [hipcc(), *HIPCC_FLAGS, "-c", src, "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{' '.join(cmd)}\n{res.stdout}\n{res.stderr}")
    return obj


def build(jobs: int | None = None, verbose: bool = False) -> str:
    os.makedirs(BUILD_DIR, exist_ok=True)
    srcs = sources()
    jobs = jobs or min(len(srcs), max(1, (os.cpu_count() or 2)))
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(_compile, srcs))
    tmp = LIB_PATH + ".tmp"
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{' '.join(cmd)}\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, LIB_PATH)
    if not _build_native() and verbose:
        print("no Python.h: _native not built, calls go through ctypes", file=sys.stderr)
    if verbose:
        print(f"built {LIB_PATH} from {len(srcs)} sources", file=sys.stderr)
    return LIB_PATH


def _build_native() -> bool:
    """Builds _native for this interpreter; those of an earlier library go, as
    their entry points may have other arguments. False without Python.h."""
    for old in glob.glob(os.path.join(HERE, "_native.*")):
        os.remove(old)
    include = sysconfig.get_paths()["include"]
    if not os.path.exists(os.path.join(include, "Python.h")):
        return False
    tmp = NATIVE_PATH + ".tmp"
    cmd = [hipcc(), "-x", "c++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Wl,--as-needed",
           "-I" + include, os.path.join(CSRC, "pycall.cpp"), "-o", tmp,
           "-L" + HERE, "-lopengenie_amd", "-Wl,-rpath,$ORIGIN"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"_native failed:\n{' '.join(cmd)}\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, NATIVE_PATH)
    return True


def main() -> None:
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=None)
    args = ap.parse_args()
    build(args.jobs, verbose=True)


if __name__ == "__main__":
    main()
