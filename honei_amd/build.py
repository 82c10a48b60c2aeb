"""Build libhsolve.so (gfx950) in-tree with hipcc, and the CPython module
_calls over it with a C compiler (left out where the interpreter's headers or
the compiler are missing: the package then makes those calls through ctypes).

Every HIP translation unit is compiled with
  --offload-arch=gfx950 -O3 -ffp-contract=off
  -Xclang -target-feature -Xclang -packed-fp32-ops
(-ffp-contract=off keeps products and sums separately rounded, as in
HONEI's tags::CPU loops; the packed-FP32 feature is switched off so no
v_pk_*_f32 forms are generated).
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libhsolve.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

SOURCES = ["ops.hip", "ell.hip", "solvers.hip", "mg_engine.hip", "mg_solve.hip", "serve.hip", "mrhs.hip", "csr.hip"]

COMMON = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", os.path.join(ROOT, "include"), "-I", CSRC, "-I", os.path.join(HERE, "include"),
    "-Wall", "-Wno-unused-result", "-Wno-unused-function",
]


def _compile(src: str) -> str:
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC, *COMMON, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    return obj


def build_calls(where: str = HERE, verbose: bool = True) -> str | None:
    """The module for this interpreter (its name carries the ABI tag); None where it cannot be built."""
    include = sysconfig.get_paths()["include"]
    cc = shutil.which("gcc") or shutil.which("cc")
    out = os.path.join(where, "_calls" + sysconfig.get_config_var("EXT_SUFFIX"))
    untagged = os.path.join(where, "_calls.so")
    for old in (out, untagged):
        if os.path.exists(old):
            os.remove(old)
    if cc is None or not os.path.exists(os.path.join(include, "Python.h")):
        if verbose:
            print(f"no C compiler or no Python.h in {include}: short calls go through ctypes")
        return None
    tmp = out + ".tmp"
    cmd = [cc, "-O2", "-std=c11", "-Wall", "-shared", "-fPIC", "-I", include, "-I", os.path.join(ROOT, "include"),
           os.path.join(CSRC, "pycalls.c"), "-L", HERE, "-l:libhsolve.so", "-Wl,-rpath,$ORIGIN",
           "-Wl,-rpath-link,/opt/rocm/lib", "-o", tmp]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"_calls failed:\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, out)
    return out


def build(verbose: bool = True) -> str:
    os.makedirs(BUILD, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=min(len(SOURCES), 4)) as ex:
        objs = list(ex.map(_compile, SOURCES))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    build_calls(verbose=verbose)
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build()
    sys.exit(0)
