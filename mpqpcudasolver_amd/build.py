"""Builds libmpqp_hip.so for gfx950 with hipcc (in-tree, next to this file)."""
from __future__ import annotations

import os
import shutil
import subprocess
import tempfile
from concurrent.futures import ThreadPoolExecutor

_DIR = os.path.dirname(os.path.abspath(__file__))
_CSRC = os.path.join(_DIR, "csrc")
# (source, extra flags): the library's host code and small kernels, then the
# groups of optimality kernels (csrc/opt_fn.hpp), longest compilations first
UNITS = [(os.path.join(_CSRC, "opt_fn.hip"), [f"-DMPQP_PART={p}"]) for p in (2, 3, 6, 7, 1, 0, 13, 12, 5, 4, 11, 10, 9, 8, 19, 18, 17, 16, 15, 14, 22, 21, 20)] + [
    (os.path.join(_CSRC, "mpqp_hip.hip"), [])]
OUT = os.path.join(_DIR, "libmpqp_hip.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    # the kernels' arithmetic is specified operation by operation: no fusion
    # beyond the explicit fma() calls
    "-ffp-contract=off",
    # no packed FP32 instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def hipcc() -> str:
    for c in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if c and os.path.exists(c):
            return c
    raise RuntimeError("hipcc not found")


def _run(cmd: list[str], verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed ({r.returncode}):\n{r.stderr[-8000:]}")


def build(verbose: bool = False, extra_flags: list[str] | None = None) -> str:
    """Compiles the HIP sources side by side and links libmpqp_hip.so;
    returns its path."""
    compile_flags = [f for f in HIPCC_FLAGS if f != "-shared"]
    workers = max(1, min(len(UNITS), int(os.environ.get("MAX_JOBS") or os.cpu_count() or 1)))
    with tempfile.TemporaryDirectory() as tmp, ThreadPoolExecutor(workers) as pool:
        objs = [os.path.join(tmp, f"unit{i}.o") for i in range(len(UNITS))]
        jobs = [pool.submit(_run, [hipcc(), *compile_flags, *flags, *(extra_flags or []), "-c", "-o", obj, src], verbose)
                for obj, (src, flags) in zip(objs, UNITS)]
        for j in jobs:
            j.result()
        out = OUT + ".tmp"
        _run([hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", out, *objs], verbose)
    os.replace(out, OUT)
    return OUT


if __name__ == "__main__":
    print(build(verbose=True))
