"""Builds libaxn_gfx950.so (the product library) and libaxn_probe_gfx950.so (streaming
yardsticks for benchmarks, include/axn_probe.h) from the HIP sources in this directory, and
axn_fast.so (fast.cpp), the host side of the usual Linear calls, with the host compiler
against the headers of the PyTorch that imports it.

    python -m axonn_amd.csrc.build

hipcc cross-compiles for gfx950 without a GPU.  The library links against the
HIP runtime by soname only, so inside a PyTorch process it binds to the HIP
runtime PyTorch has already loaded.
"""

import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
LIB_DIR = os.path.join(os.path.dirname(HERE), "lib")
LIB_PATH = os.path.join(LIB_DIR, "libaxn_gfx950.so")
PROBE_LIB_PATH = os.path.join(LIB_DIR, "libaxn_probe_gfx950.so")
FAST_PATH = os.path.join(LIB_DIR, "axn_fast.so")
OBJ_DIR = os.path.join(HERE, "build")

SOURCES = ["axn_api.hip", "gemm_bf16.hip", "gemm_edge_bf16.hip", "gemm_edge_f16.hip",
           "gemm_fed_nt_bf16.hip", "gemm_fed_nt_f16.hip", "gemm_fed_nn_tn_bf16.hip", "gemm_fed_nn_tn_f16.hip", "gemm_fed_rounds.hip",
           "gemm_gate_up.hip",
           "gemm_stream.hip", "gemm_far.hip", "gemm_f32.hip", "elementwise.hip", "embedding.hip", "optim.hip"]
PROBE_SOURCES = ["stream_probe.hip"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fvisibility=hidden",
    "-Wall",
    "-Wno-unused-function",
    # packed fp32 VALU forms are kept out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I" + os.path.join(ROOT, "include"),
    "-I" + HERE,
]


def _run(cmd):
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    # hipcc's host pass does not know the packed-fp32 feature name; that warning is noise.
    out = "\n".join(
        line for line in proc.stdout.splitlines()
        if "packed-fp32-ops" not in line
    )
    if proc.returncode != 0:
        raise RuntimeError("command failed: %s\n%s" % (" ".join(cmd), out))
    return out


def build_fast():
    """Compiles and links axn_fast.so.  Its libraries are PyTorch's, found by soname in the process that has them."""
    import torch

    from .._native import fast_built_for

    base = os.path.dirname(torch.__file__)
    tmp = FAST_PATH + ".tmp"
    _run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
          "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch.compiled_with_cxx11_abi(),
          '-DAXN_BUILT_FOR="%s"' % fast_built_for(torch), *("-isystem" + d for d in (os.path.join(base, "include"), os.path.join(base, "include", "torch", "csrc", "api", "include"),
                                     os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"),
                                     sysconfig.get_paths()["include"])),
          "-I" + os.path.join(ROOT, "include"), os.path.join(HERE, "fast.cpp"), "-o", tmp, "-L" + os.path.join(base, "lib"),
          "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"])
    os.replace(tmp, FAST_PATH)   # (a running process keeps the file it has mapped)


def build_fast_if_possible():
    """The package works without axn_fast.so: without a host compiler, or PyTorch's headers, the library alone is built."""
    try:
        build_fast()
    except (ImportError, OSError, RuntimeError) as error:
        if os.path.exists(FAST_PATH):
            os.remove(FAST_PATH)   # (what is left of an earlier build is of other sources)
        print("axn_fast.so is not built, Linear calls will take more host time: %s" % error, file=sys.stderr)


def build_library(verbose=False, extra_flags=()):
    """Compiles every source and links the shared library; returns its path."""
    os.makedirs(LIB_DIR, exist_ok=True)
    os.makedirs(OBJ_DIR, exist_ok=True)

    def compile_one(src):
        obj = os.path.join(OBJ_DIR, os.path.splitext(src)[0] + ".o")
        out = _run([HIPCC, *FLAGS, *extra_flags, "-c", os.path.join(HERE, src), "-o", obj])
        if verbose and out.strip():
            print(out)
        return obj

    every = SOURCES + PROBE_SOURCES
    with ThreadPoolExecutor(max_workers=min(len(every) + 1, os.cpu_count() or 1)) as pool:
        fast = pool.submit(build_fast_if_possible)
        objs = list(pool.map(compile_one, every))
        fast.result()
    for path, part in ((LIB_PATH, objs[:len(SOURCES)]), (PROBE_LIB_PATH, objs[len(SOURCES):])):
        out = _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", *part, "-o", path])
        if verbose and out.strip():
            print(out)
    return LIB_PATH


if __name__ == "__main__":
    path = build_library(verbose=True)
    print("built", path)
    sys.exit(0)
