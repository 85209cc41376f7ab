"""Builds libcfd_amd.so (HIP, gfx950) in-tree, and the test-side oracle
libraries when asked.

    python -m cfd_amd.build            # library only
    python -m cfd_amd.build --all      # + oracle/liboracle.so (+ oracle/_ref)
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
OBJ = os.path.join(PKG, "_build")
LIB = os.path.join(PKG, "libcfd_amd.so")
SOURCES = ["tables.hip", "geom.hip", "flow.hip", "pcg.hip", "patches.hip", "mlp.hip",
           "warmstart.hip", "state.hip", "batch.hip", "api.hip", "restart.hip",
           "smooth.hip"]
HEADERS = ["cfd_internal.hpp", "reduce.hpp", "crmath.hpp", "stepctl.hpp", "forces.hpp"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
# -ffp-contract=off: products and sums stay separately rounded, as in the
# reference build; packed FP32 ops are disabled for all device code.
HIP_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-fPIC", "-std=c++17", "-ffp-contract=off",
    "-fno-gpu-rdc", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-result",
]


def _newer(target: str, deps: list[str]) -> bool:
    if not os.path.exists(target):
        return True
    t = os.path.getmtime(target)
    return any(os.path.getmtime(d) > t for d in deps)


def _run(cmd: list[str]) -> None:
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("build step failed: " + " ".join(cmd[:3]) + " ...")
    # keep warnings visible but compact
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
    if err.strip():
        sys.stderr.write(err + "\n")


def build_library(force: bool = True, jobs: int = 8) -> str:
    os.makedirs(OBJ, exist_ok=True)
    hdrs = [os.path.join(CSRC, h) for h in HEADERS] + [os.path.join(ROOT, "include", "cfd_abi.h")]
    objs, todo = [], []
    for src in SOURCES:
        sp = os.path.join(CSRC, src)
        op = os.path.join(OBJ, src.replace(".hip", ".o"))
        objs.append(op)
        if force or _newer(op, [sp] + hdrs):
            todo.append([HIPCC, *HIP_FLAGS, "-c", sp, "-o", op])
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        list(ex.map(_run, todo))
    tmp = LIB + ".tmp"
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp])
    os.replace(tmp, LIB)
    return LIB


FORTRAN = os.path.join(PKG, "fortran")
ABI_DEMO = os.path.join(OBJ, "abi_demo")
SESSION_DEMO = os.path.join(OBJ, "session_demo")


def build_fortran() -> str | None:
    """The Fortran interface module (cfd_amd/fortran/cfd_abi.f90) and the demo
    driver that calls the library through it, linked against libcfd_amd.so
    (found next to the package at run time).  None when flang is absent."""
    fc = shutil.which("flang")
    if fc is None:
        return None
    os.makedirs(OBJ, exist_ok=True)
    abi_o = os.path.join(OBJ, "cfd_abi_f.o")
    _run([fc, "-O2", "-J", OBJ, "-c", os.path.join(FORTRAN, "cfd_abi.f90"), "-o", abi_o])
    for prog, exe in (("abi_demo", ABI_DEMO), ("session_demo", SESSION_DEMO)):
        obj = os.path.join(OBJ, prog + "_f.o")
        _run([fc, "-O2", "-J", OBJ, "-c", os.path.join(FORTRAN, prog + ".f90"), "-o", obj])
        _run([fc, obj, abi_o, "-L" + PKG, "-lcfd_amd", "-Wl,-rpath,$ORIGIN/..", "-o", exe])
    return ABI_DEMO


def build_oracle() -> None:
    _run(["make", "-s", "-C", ROOT, "-f", "oracle/Makefile"])


def build_reference() -> bool:
    """Compiles the reference into oracle/_ref when its sources are present,
    and the Fortran shims against the reference's own module sources."""
    if not os.path.isfile("/root/reference/mLaplace.f90") or shutil.which("flang") is None:
        return False
    _run(["make", "-s", "-C", ROOT, "-f", "oracle/Makefile.ref", "all", "shims", "shimharness"])
    return True


if __name__ == "__main__":
    build_library(force="--incremental" not in sys.argv)
    build_fortran()
    if "--all" in sys.argv:
        build_oracle()
        build_reference()
    print(LIB)
