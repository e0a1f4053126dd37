"""Build recipe for the native libraries of cpw2000_amd (in-tree).

  libcpwgpu.so          HIP kernels + C ABI (include/cpwgpu.h), gfx950
  libcpwgpu_fortran.so  Fortran drop-ins hk_psi_c16, hk_psi_spin_c16 and ditsp_c16, and the all-k
                        hk_psi_allk_c16, over the C ABI (flang)
  libcpwprobe.so        VALU issue-rate probe (measurement only: ``bench.py --issue-rates``)

Run ``python -m cpw2000_amd.build``.
"""

from __future__ import annotations

import os
import re
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
LIB = os.path.join(PKG, "libcpwgpu.so")
FLIB = os.path.join(PKG, "libcpwgpu_fortran.so")
OBJ = os.path.join(ROOT, "build")
PLIB = os.path.join(PKG, "libcpwprobe.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLANG = os.environ.get("FLANG", shutil.which("flang") or "/opt/rocm/lib/llvm/bin/flang")
ARCH = os.environ.get("CPWGPU_ARCH", "gfx950")

HIP_FLAGS = [
    "-O3", "-std=c++17", f"--offload-arch={ARCH}", "-fPIC",
    # no packed FP32 instructions anywhere in device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
]


def _run(cmd):
    print("+", " ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)


def mesh_lengths(which="CPW_FAST_SIZES"):
    """The specialised mesh lengths (CPW_FAST_SIZES or CPW_FULL_SIZES of csrc/mesh.hpp)."""
    with open(os.path.join(CSRC, "mesh.hpp")) as f:
        line = next(t for t in f if t.startswith("#define " + which))
    return [int(n) for n in re.findall(r"X\((\d+)\)", line)]


def build_hip():
    # one object per specialised mesh length (csrc/mesh.hip), side by side, and
    # the rest (csrc/cpwgpu.hip); the longest compiles first
    os.makedirs(OBJ, exist_ok=True)
    jobs = [("cpwgpu.hip", "cpwgpu.o", [])]
    full = mesh_lengths("CPW_FULL_SIZES")
    jobs += [("mesh.hip", f"mesh{n}.o", [f"-DCPW_N={n}", f"-DCPW_N_FULL={int(n in full)}"])
             for n in sorted(mesh_lengths(), key=lambda n: (n in full, n), reverse=True)]
    objs = [os.path.join(OBJ, o) for _, o, _ in jobs]

    def compile_one(job):
        src, obj, defs = job
        _run([HIPCC, *HIP_FLAGS, "-c", *defs, "-I", os.path.join(ROOT, "include"), "-o", os.path.join(OBJ, obj),
              os.path.join(CSRC, src)])

    with ThreadPoolExecutor(max_workers=int(os.environ.get("MAX_JOBS", 0)) or os.cpu_count() or 1) as pool:
        for done in [pool.submit(compile_one, j) for j in jobs]:
            done.result()
    tmp = LIB + ".tmp"
    # rocSOLVER (zheevd, zpotrf) and rocBLAS (ztrsm) for the small dense
    # eigenproblems of the iterative diagonalisation.  The first device bundle
    # of the library is the one that offload tools read: length 72, which has
    # every kind of line transform.
    objs.sort(key=lambda o: not o.endswith("mesh72.o"))
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-o", tmp, *objs, "-lrocsolver", "-lrocblas"])
    os.replace(tmp, LIB)


def build_probe():
    tmp = PLIB + ".tmp"
    _run([HIPCC, *HIP_FLAGS, "-shared", "-o", tmp, os.path.join(CSRC, "issue_rates.hip")])
    os.replace(tmp, PLIB)


def build_fortran():
    srcs = [os.path.join(PKG, "fortran", f)
            for f in ("hk_psi_c16.f90", "hk_psi_spin_c16.f90", "ditsp_c16.f90", "hk_psi_allk_c16.f90",
                      "proj_nl_kb_c16.f90")]
    tmp = FLIB + ".tmp"
    objdir = os.path.join(PKG, "fortran")
    _run([FLANG, "-O2", "-fPIC", "-shared", "-module-dir", objdir, "-o", tmp, *srcs,
          "-L", PKG, "-lcpwgpu", "-Wl,-rpath,$ORIGIN"])
    os.replace(tmp, FLIB)


def build(fortran: bool = True):
    build_hip()
    build_probe()
    if fortran:
        build_fortran()


if __name__ == "__main__":
    build(fortran="--no-fortran" not in sys.argv)
