"""Build recipe of libfusor_hip.so: every .hip file of csrc/ compiled for gfx950 and linked into one
shared library beside this file.  Run as `python -m kalosm_amd.build` or through `__graft_entry__.build()`."""
from __future__ import annotations

import fcntl
import glob
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
LIB = os.path.join(HERE, "libfusor_hip.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",          # dequantised values are compared bit for bit: never fuse a*b - c
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unknown-warning-option", "-Wno-unused-command-line-argument",
    "-fvisibility=hidden",
]
AHEAD = ["-mllvm", "-amdgpu-kernarg-preload-count=14"]  # the first words of a kernel's plain arguments are in registers when it starts
# Arguments are loaded ahead only where the first requests need no others: prompt attention's need three pointers and nine strides
# (8 heads of 128, 300 tokens: 10.18 us without, 10.25 with).
LOADS_ARGUMENTS = {"fh_attention_prefill.hip"}


def _compile(src: str) -> str:
    obj = os.path.join(OBJ, os.path.basename(src) + ".o")
    ahead = [] if os.path.basename(src) in LOADS_ARGUMENTS else AHEAD
    cmd = [HIPCC, *FLAGS, *ahead, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stdout}\n{r.stderr}")
    warn = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l and l.strip())
    if warn:
        sys.stderr.write(warn + "\n")
    return obj


def build(jobs: int = 8, verbose: bool = True) -> str:
    os.makedirs(OBJ, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    if not srcs:
        raise RuntimeError("no sources under " + CSRC)
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(_compile, srcs))
    part = LIB + f".{os.getpid()}"
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", part, *objs, "-Wl,--no-undefined"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(part, LIB)
    if verbose:
        print(f"built {LIB} from {len(srcs)} sources")
    return LIB


def ensure() -> str:
    """The library, built first when it is not there (one process builds, others wait)."""
    if not os.path.exists(LIB):
        with open(os.path.join(HERE, ".build.lock"), "w") as lock:
            fcntl.flock(lock, fcntl.LOCK_EX)
            if not os.path.exists(LIB):
                build(jobs=min(16, os.cpu_count() or 1), verbose=False)
    return LIB


if __name__ == "__main__":
    build()
