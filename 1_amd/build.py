"""Build recipe for libgpukern.so (gfx950).

Compiles every HIP translation unit under ``csrc/`` with hipcc in parallel and
links them into ``1_amd/libgpukern.so``.  Run directly (``python 1_amd/build.py``)
or through ``__graft_entry__.build()``.
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libgpukern.so")

SOURCES = ["gk_basic.hip", "gk_fft.hip", "gk_fft_any.hip", "conv.hip", "rk.hip", "sim.hip", "batch.hip", "io.cpp"]
# kernels with many length instantiations, compiled in parts (-DGK_PART=i): they set the build's time
PARTS = {"conv_z.hip": 7, "batch_z.hip": 7, "batch_any.hip": 4}

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # packed FP32 instructions are kept out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def _compile(job):
    src, part = job
    name = os.path.splitext(src)[0] + ("" if part is None else "_%d" % part)
    obj = os.path.join(BUILD, name + ".o")
    defs = [] if part is None else ["-DGK_PART=%d" % part]
    cmd = [HIPCC, *FLAGS, *defs, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    msgs = [l for l in (r.stdout + r.stderr).splitlines() if "packed-fp32" not in l and "warning: feature" not in l]
    if r.returncode != 0:
        raise RuntimeError("hipcc failed for %s:\n%s" % (src, "\n".join(msgs)))
    return obj


def build(verbose=False):
    os.makedirs(BUILD, exist_ok=True)
    # the longest first: the conv_z parts, the dispatch kernels of the Z inverse, batch and conv
    jobs = [(src, i) for src, n in PARTS.items() for i in range(n)] + [(src, None) for src in SOURCES]
    slow = {"conv_z.hip": 0, "batch.hip": 1, "conv.hip": 1, "batch_any.hip": 2, "batch_z.hip": 3}
    jobs.sort(key=lambda j: slow.get(j[0], 4))
    with ThreadPoolExecutor(max_workers=min(len(jobs), os.cpu_count() or 4)) as ex:
        objs = list(ex.map(_compile, jobs))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stdout + r.stderr)
    os.replace(tmp, LIB)
    if verbose:
        print("built", LIB)
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
