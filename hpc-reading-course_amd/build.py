"""Build recipe of the HIP library (gfx950) and the demo drivers.

Compiles every csrc/*.hip translation unit with hipcc in parallel and links
libsbp_hip.so in this directory (in-tree, so it travels with the repository
snapshot).  Objects go to _build/.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libsbp_hip.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
HIPFLAGS = ["--offload-arch=" + ARCH, "-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function",
            "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def _run(cmd):
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in r.stdout.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError("command failed (%d): %s\n%s" % (r.returncode, " ".join(cmd), out))
    return out


def extra_flags(src):
    # Solver kernels: no FMA contraction.  FP64 right-hand sides round exactly
    # like the reference's loops (mul then add, in the same order), and FP32
    # multiply-adds are fused where the source says so (sbp_kernels.hpp mad), the
    # same way in every kernel.
    if src.endswith(("_f64.hip", "_f32.hip")):
        return ["-ffp-contract=off"]
    # The corrector's MFMA kernels keep their accumulators in ordinary VGPRs
    # (no AGPR copies before the bias/ReLU/bf16 epilogues); the occupancy of
    # every kernel in the file is the same either way.
    if src.endswith("sbp_corr.hip"):
        return ["-mllvm", "-amdgpu-mfma-vgpr-form"]
    return []


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def build(jobs: int | None = None, verbose: bool = False) -> str:
    os.makedirs(OBJ, exist_ok=True)
    srcs = sources()
    objs = [os.path.join(OBJ, os.path.basename(s)[:-4] + ".o") for s in srcs]
    jobs = jobs or min(8, os.cpu_count() or 4)
    with cf.ThreadPoolExecutor(jobs) as ex:
        futs = [ex.submit(_run, [HIPCC, *HIPFLAGS, *extra_flags(s), "-c", s, "-o", o])
                for s, o in zip(srcs, objs)]
        for f in futs:
            msg = f.result()
            if verbose and msg.strip():
                print(msg)
    tmp = LIB + ".tmp"
    _run([HIPCC, "--offload-arch=" + ARCH, "-shared", "-fPIC", "-o", tmp, *objs])
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
