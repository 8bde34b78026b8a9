"""Builds the HIP library (libtensornet_amd.so) in-tree with hipcc for gfx950, and the Python
binding of its operators (_bind.so).

    python -m tensornet_amd.build

hipcc cross-compiles without a GPU.  The flags keep fp32 arithmetic IEEE
(no FMA contraction, correctly rounded divide / sqrt) so that optimizer
updates can be compared element for element with a CPU evaluation, and turn
packed-fp32 instruction selection off.
"""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libtensornet_amd.so")
SOURCES = ["core.hip", "dense_table.hip", "sparse_table.hip", "checkpoint.hip"]
KIND_SOURCE = "apply_kind.hip"  # compiled once per optimizer (AdaGrad, Adam, Ftrl)

FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
]


BIND_SRC = os.path.join(CSRC, "bind.cc")
BIND = os.path.join(HERE, "_bind.so")

HOST_TEST_SRC = os.path.join(ROOT, "tests", "cpp", "host_mirror_test.cc")
HOST_TEST_BIN = os.path.join(ROOT, "tests", "cpp", "host_mirror_test")


def build(verbose=True):
    """Compiles the sources side by side (most of the time goes to sparse_table.hip), then links them."""
    import tempfile
    from concurrent.futures import ThreadPoolExecutor

    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    units = [(s, []) for s in SOURCES] + [(KIND_SOURCE, ["-DTN_KIND=%d" % k]) for k in range(3)]

    def run(cmd):
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.check_call(cmd)

    with tempfile.TemporaryDirectory() as tmp:
        def compile_unit(i):
            source, defines = units[i]
            obj = os.path.join(tmp, "%d.o" % i)
            run([hipcc] + FLAGS + defines + ["-I", os.path.join(ROOT, "include"), "-I", CSRC, "-c", os.path.join(CSRC, source), "-o", obj])
            return obj

        with ThreadPoolExecutor(min(len(units), int(os.environ.get("MAX_JOBS", "8")))) as pool:
            objs = list(pool.map(compile_unit, range(len(units))))
        run([hipcc, "--offload-arch=gfx950", "-fPIC", "-shared"] + objs + ["-lz", "-o", LIB])
    return LIB


def build_bind(verbose=True):
    """Builds the Python binding of the operators (host code over torch's C++ headers, linked to the library)."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths, library_paths

    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM=1", "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI,
           "-I", os.path.join(ROOT, "include"), "-I", os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"),
           "-I", sysconfig.get_paths()["include"]]
    cmd += [a for p in include_paths() for a in ("-isystem", p)]
    cmd += [BIND_SRC, "-o", BIND, "-L", HERE, "-ltensornet_amd", "-Wl,-rpath,$ORIGIN"]
    cmd += [a for p in library_paths() for a in ("-L", p)] + ["-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    return BIND


def build_host_test(verbose=True):
    """Builds the C++ program that drives the library through include/tensornet_amd.hpp."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    cmd = [hipcc, "-std=c++17", "-O1", "-I", os.path.join(ROOT, "include"), HOST_TEST_SRC, "-L", HERE,
           "-ltensornet_amd", "-Wl,-rpath,$ORIGIN/../../tensornet_amd", "-o", HOST_TEST_BIN]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    return HOST_TEST_BIN


if __name__ == "__main__":
    build()
    build_bind()
    build_host_test()
    sys.exit(0)
