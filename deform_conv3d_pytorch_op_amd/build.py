"""Builds csrc/libdcn_amd.so with hipcc for gfx950 (in-tree, no JIT cache).  The translation units
compile side by side.

    python -m deform_conv3d_pytorch_op_amd.build
"""
import glob
import os
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
SO = os.path.join(CSRC, "libdcn_amd.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # packed fp32 math is switched off on purpose for this target
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # float/double atomic adds lower to global_atomic_add_f32/f64 instead of CAS loops
    "-munsafe-fp-atomics",
]


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in r.stdout.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError("hipcc failed:\n" + out)
    if verbose and out.strip():
        print(out)


def build(verbose=False):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    sources = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    jobs = min(len(sources), int(os.environ.get("MAX_JOBS", 0) or os.cpu_count() or 1))
    with tempfile.TemporaryDirectory() as tmp:
        objects = [os.path.join(tmp, os.path.basename(s) + ".o") for s in sources]
        with ThreadPoolExecutor(jobs) as pool:
            list(pool.map(lambda so: _run([hipcc] + HIPCC_FLAGS + ["-c", "-o", so[1], so[0]], verbose), zip(sources, objects)))
        _run([hipcc] + HIPCC_FLAGS + ["-shared", "-o", SO] + objects, verbose)
    return SO


if __name__ == "__main__":
    print(build(verbose=True))
    sys.exit(0)
