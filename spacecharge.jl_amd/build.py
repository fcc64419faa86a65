"""Build libspacecharge_mi355.so (gfx950) in-tree with hipcc.

Usage: python spacecharge.jl_amd/build.py   (or spacecharge.build_library())

Every translation unit under csrc/ is compiled for gfx950 only, then linked
into one shared library next to this file.  Flags:
  -munsafe-fp-atomics   hardware float/double atomic adds for the deposit
  -Xclang -target-feature -Xclang -packed-fp32-ops
                        no packed-FP32 instructions in generated code
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(REPO, "include")
OBJDIR = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libspacecharge_mi355.so")
ARCH = "gfx950"

# (source, object suffix, extra flags); the transform kernels, one set per
# length and mesh type, compile in parts that build in parallel
UNITS = [("sc_solve_mix.hip", f"_{k}", [f"-DSC_MIX_PART={k}"]) for k in range(4)]
UNITS += [("sc_green.hip", f"_{k}", [f"-DSC_GREEN_PART={k}"]) for k in range(2)]
UNITS += [("sc_solve_plane.hip", f"_{k}", [f"-DSC_PLANE_PART={k}"]) for k in range(2)]
UNITS += [("sc_api.cpp", "", []), ("sc_particles.hip", "", []), ("sc_deposit.hip", "", []),
          ("sc_solve.hip", "", []), ("sc_solve_fast.hip", "", [])]
HEADERS = ["sc_internal.h", "sc_deposit_plan.h", "sc_fft_dev.h", "sc_fft_reg.h", "sc_fft_mix.h",
           "sc_solve_common.h"]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (ROCm is required to build the library)")


COMMON = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-munsafe-fp-atomics",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-result",
    f"-I{INCLUDE}",
    f"-I{CSRC}",
]


def _compile(unit) -> str:
    src, suffix, flags = unit
    obj = os.path.join(OBJDIR, os.path.splitext(src)[0] + suffix + ".o")
    cmd = [hipcc()] + COMMON + flags + ["-c", os.path.join(CSRC, src), "-o", obj]
    if src.endswith(".cpp"):
        cmd[1:1] = ["-x", "hip"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{r.stderr}")
    return obj


def build(verbose: bool = False) -> str:
    """Compile every source (always) and link the shared library; returns its path."""
    os.makedirs(OBJDIR, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=min(len(UNITS), os.cpu_count() or 1)) as ex:
        objs = list(ex.map(_compile, UNITS))
    tmp = LIB + ".tmp"
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
