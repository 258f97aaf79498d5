"""Build the gfx950 shared library of the expert hot path in-tree.

    python -m moe_stream_amd.build

writes moe_stream_amd/lib/libmoe_stream.so with hipcc.  The library links the
HIP runtime by soname (libamdhip64.so.7); loaded after `import torch` it binds
to the runtime torch already holds, so one HIP runtime is in the process.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
LIBDIR = PKG / "lib"
LIB = LIBDIR / "libmoe_stream.so"
ARCH = os.environ.get("MOE_OFFLOAD_ARCH", "gfx950")

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    # no packed fp32 instructions anywhere in device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # MFMA results straight into VGPRs (no accumulator-register copies).
    # Chained MFMAs may then read an accumulator input apart from their
    # destination, and whatever writes that input next must stay clear of them.
    # In the built assembly no compiler-made instruction comes closer than 4
    # issue slots to a bf16 MFMA that reads the register; instructions written
    # as inline asm, which the compiler does not look into, come as close as 1.
    # (To an fp32 MFMA that reads one, compiler-made ones come as close as 1.)  So
    # the MFMA kernels decode codes with ordinary operations, their asm statements
    # are empty, and their fp32 MFMAs start from zero.
    "-Xarch_device", "-mllvm=-amdgpu-mfma-vgpr-form=1",
    "-Wno-unused-command-line-argument",
]


def hipcc() -> str:
    for c in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if c and Path(c).exists():
            return c
    raise RuntimeError("hipcc not found; the HIP library cannot be built")


def build(verbose: bool = True) -> Path:
    LIBDIR.mkdir(exist_ok=True)
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [hipcc(), *HIPCC_FLAGS, "-I", str(PKG.parent / "include"),
           str(CSRC / "libmoe_stream.hip"), "-o", str(tmp)]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in r.stderr.splitlines() if noise not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed ({r.returncode}):\n{err}")
    if verbose and err.strip():
        print(err, file=sys.stderr)
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build())
