"""Build libmegaslide_dsa3d.so for gfx950 with hipcc, in-tree.

    python -m megaslide_amd.csrc.build          # or: python megaslide_amd/csrc/build.py

Each .hip source is compiled to an object (in parallel), then linked into
megaslide_amd/lib/libmegaslide_dsa3d.so.  The library links libamdhip64.so.7
by soname, so inside a process that imported torch it binds to the HIP
runtime torch already loaded.
"""

from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.dirname(HERE)
ROOT = os.path.dirname(PKG)
LIB_DIR = os.path.join(PKG, "lib")
LIB_NAME = "libmegaslide_dsa3d.so"
OBJ_DIR = os.path.join(ROOT, "_build", "obj")

SOURCES = ["abi.hip", "dsa3d_direct.hip", "dsa3d_fwd.hip", "dsa3d_ragged.hip",
           "dsa3d_bwd1.hip", "dsa3d_tiled.hip", "dwconv3d.hip"]

ARCH = os.environ.get("MSD_OFFLOAD_ARCH", "gfx950")

CFLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++20",
    "-fPIC",
    "-munsafe-fp-atomics",
    # packed fp32 instructions stay off: ordinary float code only
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
    "-I", os.path.join(ROOT, "include"),
    "-I", HERE,
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (ROCm toolchain required to build the HIP library)")


def _compile(src: str) -> str:
    obj = os.path.join(OBJ_DIR, os.path.splitext(src)[0] + ".o")
    cmd = [hipcc(), *CFLAGS, "-c", os.path.join(HERE, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{r.stderr}")
    return obj


def build(verbose: bool = False) -> str:
    os.makedirs(OBJ_DIR, exist_ok=True)
    os.makedirs(LIB_DIR, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=min(len(SOURCES), os.cpu_count() or 1)) as ex:
        objs = list(ex.map(_compile, SOURCES))
    out = os.path.join(LIB_DIR, LIB_NAME)
    tmp = out + ".tmp"
    # -z defs: every symbol resolved at link time (a kernel whose host-side
    # launch stub was not emitted would otherwise only fail when loaded)
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-Wl,-z,defs", *objs, "-o", tmp]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(tmp, out)
    if verbose:
        print("built", out)
    return out


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
