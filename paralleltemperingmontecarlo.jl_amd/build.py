"""Build libptmc.so (HIP, gfx950) in-tree.

    python paralleltemperingmontecarlo.jl_amd/build.py

Each csrc/*.hip is compiled to an object under _build/ in parallel and the
objects are linked into lib/libptmc.so next to this file.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import pathlib
import shutil
import subprocess
import sys

HERE = pathlib.Path(__file__).resolve().parent
CSRC = HERE / "csrc"
BUILD = HERE / "_build"
LIB = HERE / "lib" / "libptmc.so"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("PTMC_OFFLOAD_ARCH", "gfx950")

# -ffp-contract=off: every fused multiply-add in the kernels is written out
# explicitly, so FP64 results are reproducible operation by operation.
# Packed FP32 instructions are disabled for all device code.
CFLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


# The moves of the network potentials run as one long loop with many phases:
# constants of every phase's polynomials hoisted out of it spill to scratch
# (VGPRs spilled with hoisting / without: two species in FP64 on 1024 threads 124
# / 25, with general powers 202 / 51; one species 19 / 0, 128-atom slots 33 / 4).
NO_MACHINE_LICM = ("ptmc_nnp", "ptmc_nnp2_mc", "ptmc_nnp2_mc_f32", "ptmc_nnp2_mc_half", "ptmc_nnp2_mc_f32_half")


def _compile(src: pathlib.Path) -> tuple[pathlib.Path, str]:
    obj = BUILD / (src.stem + ".o")
    extra = ["-mllvm", "-disable-machine-licm"] if src.stem in NO_MACHINE_LICM else []
    cmd = [HIPCC, *CFLAGS, *extra, "-c", str(src), "-o", str(obj)]
    p = subprocess.run(cmd, capture_output=True, text=True)
    log = (p.stdout + p.stderr).strip()
    # the host pass does not know the packed-fp32 target feature; that warning is expected
    log = "\n".join(l for l in log.splitlines() if "packed-fp32-ops" not in l and "not a recognized feature" not in l)
    if p.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{log}")
    return obj, log


def build(jobs: int | None = None, verbose: bool = False) -> pathlib.Path:
    if not shutil.which(HIPCC) and not os.path.exists(HIPCC):
        raise RuntimeError(f"hipcc not found at {HIPCC}")
    BUILD.mkdir(exist_ok=True)
    LIB.parent.mkdir(exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    jobs = jobs or min(8, os.cpu_count() or 1, len(sources))
    objs = []
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        for obj, log in ex.map(_compile, sources):
            objs.append(obj)
            if verbose and log:
                print(log, file=sys.stderr)
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    p = subprocess.run(cmd, capture_output=True, text=True)
    if p.returncode != 0:
        raise RuntimeError(f"link failed: {' '.join(cmd)}\n{p.stdout}{p.stderr}")
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    path = build(verbose="-v" in sys.argv)
    print(path)
