"""Builds csrc/libdcn_amd.so with hipcc for gfx950 and the C++ extension _native.so on top of it
(in-tree, no JIT cache).  The translation units compile side by side.

    python -m deform_conv3d_pytorch_op_amd.build
"""
import glob
import os
import subprocess
import sys
import sysconfig
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
SO = os.path.join(CSRC, "libdcn_amd.so")
NATIVE = os.path.join(HERE, "_native.so")

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


def _torch_flags():
    import torch
    root = os.path.dirname(torch.__file__)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    include = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
               os.path.join(rocm, "include"), sysconfig.get_paths()["include"]]
    compile_flags = ["-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
                     "-D_GLIBCXX_USE_CXX11_ABI=%d" % int(torch._C._GLIBCXX_USE_CXX11_ABI)] + ["-I" + d for d in include]
    link_flags = ["-L" + os.path.join(root, "lib"), "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10", "-lc10_hip",
                  "-L" + CSRC, "-ldcn_amd", "-Wl,-rpath,$ORIGIN/csrc"]
    return compile_flags, link_flags


def build(verbose=False):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    cxx = os.environ.get("CXX", "g++")
    sources = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    jobs = min(len(sources) + 1, int(os.environ.get("MAX_JOBS", 0) or os.cpu_count() or 1))
    compile_flags, link_flags = _torch_flags()
    with tempfile.TemporaryDirectory() as tmp:
        objects = [os.path.join(tmp, os.path.basename(s) + ".o") for s in sources]
        native = os.path.join(tmp, "dcn_torch.o")
        commands = [[cxx] + compile_flags + ["-c", "-o", native, os.path.join(CSRC, "dcn_torch.cpp")]]
        commands += [[hipcc] + HIPCC_FLAGS + ["-c", "-o", o, s] for s, o in zip(sources, objects)]
        with ThreadPoolExecutor(jobs) as pool:
            list(pool.map(lambda c: _run(c, verbose), commands))
        _run([hipcc] + HIPCC_FLAGS + ["-shared", "-o", SO] + objects, verbose)
        _run([cxx, "-shared", "-o", NATIVE, native] + link_flags, verbose)
    return SO


if __name__ == "__main__":
    print(build(verbose=True))
    sys.exit(0)
