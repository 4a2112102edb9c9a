"""Build libctraj.so in-tree with hipcc for gfx950, the sources side by side."""
from __future__ import annotations

import os
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG.parent / "csrc"
INCLUDE = PKG.parent.parent / "include"
OUT = PKG / "libctraj.so"

SOURCES = ["ctraj.hip", "batch.hip", "record.hip", "adjoint.hip", "sort.hip", "resample.hip"]
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-ffp-contract=off",  # every fused multiply-add in the kernels is written out explicitly
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]
# This compiler (ROCm 7.2) has lost track of a register that it had joined with another and produced a kernel with
# wrong results.  Its own verifier, run before registers are given out, reports that as an error and ends the build
# (the slowest source: 30 s without, 100 s with it).
VERIFY = ["-mllvm", "-verify-regalloc"]


def build(out: Path = OUT, verbose: bool = False) -> Path:
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    tmp = out.with_suffix(".so.tmp")

    def run(cmd):
        if verbose:
            print(" ".join(cmd), flush=True)
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            sys.stderr.write(r.stdout + r.stderr)
            raise RuntimeError("hipcc failed")

    with tempfile.TemporaryDirectory() as d, ThreadPoolExecutor(len(SOURCES)) as pool:
        objs = [str(Path(d) / (Path(s).stem + ".o")) for s in SOURCES]
        for job in [pool.submit(run, [hipcc, *FLAGS, *VERIFY, "-I", str(INCLUDE), "-c", str(CSRC / s), "-o", o])
                    for s, o in zip(SOURCES, objs)]:
            job.result()
        run([hipcc, "--offload-arch=gfx950", "-shared", "-o", str(tmp), *objs])
    os.replace(tmp, out)
    return out


if __name__ == "__main__":
    print(build(verbose=True))
