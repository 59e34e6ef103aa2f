"""Builds the native code in-tree.

    python -m lookahead_keys_attention_amd.build

libcastle_hip.so   HIP kernels + C ABI for gfx950, with hipcc: plain HIP behind include/castle_hip.h, no torch headers
_castle_host.so    csrc/castle_host.cpp, with g++ against the torch headers: operators and host path over that ABI
"""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_NAME = "libcastle_hip.so"
LIB_PATH = os.path.join(HERE, LIB_NAME)
SOURCES = ("castle_fwd.hip", "castle_bwd.hip", "castle_narrow.hip", "castle_narrow_bwd.hip", "castle_short.hip", "castle_decode.hip", "castle_rows.hip", "castle_gemm.hip", "castle_gemm32.hip", "castle_profile.hip", "castle_abi.hip")
HOST_SOURCE = "castle_host.cpp"
HOST_NAME = "_castle_host.so"
ARCH = "gfx950"
# packed fp32 VALU instructions stay disabled on purpose (hipcc's host pass warns that it
# does not know the feature; that warning is harmless)
HIPCC_FLAGS = (
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
)
# Kernels of one wave per SIMD have 256 accumulation registers beside the vector registers, and the compiler then lets every matrix
# instruction write there, which costs a copy for each register that a vector instruction reads.  With this the results lie in vector
# registers and the other file takes what does not fit.  An internal option of the compiler: one that does not know it builds without.
VECTOR_RESULTS = ("-mllvm", "-amdgpu-mfma-vgpr-form=1")
SOURCE_FLAGS = {"castle_narrow.hip": VECTOR_RESULTS}


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.isabs(cand) and os.path.exists(cand) or not os.path.isabs(cand)):
            return cand
    return "hipcc"


def _host_compiler():
    import torch

    include = os.path.join(os.path.dirname(torch.__file__), "include")
    return ["g++", "-std=c++17", "-O2", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM", "-I" + include,
            "-I" + os.path.join(include, "torch", "csrc", "api", "include"), "-isystem", "/opt/rocm/include",
            "-I" + sysconfig.get_paths()["include"]]


def _run(cmd):
    proc = subprocess.run(cmd, capture_output=True, text=True)
    noise = "'-packed-fp32-ops' is not a recognized feature"
    err = "\n".join(l for l in proc.stderr.splitlines() if noise not in l and "warning" not in l.lower() or "error" in l.lower())
    if proc.returncode != 0:
        raise RuntimeError(f"command failed: {' '.join(cmd)}\n{proc.stdout}\n{proc.stderr}")
    return err


def build(verbose: bool = False, jobs: int | None = None) -> str:
    """Compile every source and link the two shared libraries; returns the path of the kernel library."""
    hipcc = _hipcc()
    objdir = os.path.join(HERE, "build")
    os.makedirs(objdir, exist_ok=True)
    jobs = jobs or min(len(SOURCES) + 1, os.cpu_count() or 1, 8)

    def compile_one(src):
        obj = os.path.join(objdir, os.path.splitext(src)[0] + ".o")
        cmd = _host_compiler() if src == HOST_SOURCE else [hipcc, *HIPCC_FLAGS]
        cmd = [*cmd, "-c", os.path.join(CSRC, src), "-o", obj]
        extra = SOURCE_FLAGS.get(src, ())
        if verbose:
            print(" ".join((*cmd, *extra)), flush=True)
        try:
            _run([*cmd, *extra])
        except RuntimeError as e:
            if not extra or "Unknown command line argument" not in str(e):
                raise
            print(f"{src}: the compiler does not know {' '.join(extra)}, compiled without", file=sys.stderr, flush=True)
            _run(cmd)
        return obj

    with ThreadPoolExecutor(max_workers=jobs) as pool:
        host_obj, *objs = pool.map(compile_one, (HOST_SOURCE, *SOURCES))
    link = [hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-fno-gpu-rdc", "-o", LIB_PATH, *objs]
    if verbose:
        print(" ".join(link), flush=True)
    _run(link)
    import torch

    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    link = ["g++", "-shared", "-o", os.path.join(HERE, HOST_NAME), host_obj, "-L" + HERE, "-lcastle_hip", "-L" + torch_lib,
            "-ltorch_python", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip", "-Wl,-rpath,$ORIGIN"]
    if verbose:
        print(" ".join(link), flush=True)
    _run(link)
    return LIB_PATH


if __name__ == "__main__":
    path = build(verbose="-q" not in sys.argv)
    print(path)
