"""Builds libsparda.so (HIP kernels for gfx950 + the C ABI) and the Python
operators' native host path in-tree.

Every HIP translation unit under ``csrc/`` is compiled by hipcc for gfx950 only,
then linked into ``sparda/libsparda.so`` next to this file; ``csrc/host.cpp``
becomes the extension module ``sparda/_host.so`` (host code alone).
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
import warnings
from concurrent.futures import ThreadPoolExecutor

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG_DIR)
CSRC = os.path.join(ROOT, "csrc")
OBJ_DIR = os.path.join(ROOT, "_build")
LIB_PATH = os.path.join(PKG_DIR, "libsparda.so")
HOST_PATH = os.path.join(PKG_DIR, "_host.so")

ARCH = "gfx950"
HIPCC = os.environ.get("HIPCC", shutil.which("hipcc") or "/opt/rocm/bin/hipcc")
FLAGS = [
    "-O3", "-std=c++17", f"--offload-arch={ARCH}", "-fPIC", "-fvisibility=hidden",
    "-Wall", "-Wno-unused-function", "-Wno-pass-failed",
    # packed fp32 VALU ops stay disabled
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(src: str) -> str:
    obj = os.path.join(OBJ_DIR, os.path.basename(src) + ".o")
    cmd = [HIPCC, *FLAGS, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    out = "\n".join(l for l in (r.stdout + r.stderr).splitlines()
                    if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{out}")
    if out.strip():
        sys.stderr.write(out + "\n")
    return obj


def _build_host() -> None:
    import torch

    t = os.path.dirname(torch.__file__)
    tmp = HOST_PATH + ".tmp"
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall", "-Wno-cast-function-type",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *(f"-isystem{d}" for d in (os.path.join(t, "include"), os.path.join(t, "include/torch/csrc/api/include"),
                                      sysconfig.get_paths()["include"])),
           os.path.join(CSRC, "host.cpp"), "-o", tmp, f"-L{os.path.join(t, 'lib')}", "-ltorch_python", "-ltorch_cpu",
           "-lc10"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed for host.cpp:\n{r.stdout}{r.stderr}")
    os.replace(tmp, HOST_PATH)


def build(jobs: int = 8) -> str:
    """Compile all HIP sources and link libsparda.so, and the host module;
    returns the library's path. A host module that cannot be built (no g++, no
    Python or torch headers) is a warning: the library does not need it, and
    the operators take their Python path."""
    os.makedirs(OBJ_DIR, exist_ok=True)
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        host = ex.submit(_build_host)
        objs = list(ex.map(_compile, sources()))
    _link(objs)
    try:
        host.result()
    except Exception as e:
        if os.path.exists(HOST_PATH):
            os.remove(HOST_PATH)  # of an earlier source
        warnings.warn(f"sparda: the native host path was not built, operators will call through Python: {e}",
                      RuntimeWarning)
    return LIB_PATH


def _link(objs) -> None:
    tmp = LIB_PATH + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-Wl,--no-undefined", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}{r.stderr}")
    os.replace(tmp, LIB_PATH)


if __name__ == "__main__":
    print(build())
