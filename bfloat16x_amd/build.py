"""Build libbf16x_hip.so (hipcc, gfx950) and _host.so in-tree.

    python -m bfloat16x_amd.build [-v]

Every HIP source is compiled for gfx950 with packed-fp32 instruction
selection disabled, host C++ sources with the same driver, and the objects
are linked into bfloat16x_amd/libbf16x_hip.so.  csrc/host_ext.cpp, the CPython
module over torch's C++ API, is compiled with g++ into bfloat16x_amd/_host.so.  Objects go to _build/
(ignored by git).
"""
from __future__ import annotations

import concurrent.futures as cf
import glob
import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "libbf16x_hip.so")
HOST_SRC = os.path.join(CSRC, "host_ext.cpp")
HOST_OUT = os.path.join(HERE, "_host.so")
BUILD_DIR = os.path.join(ROOT, "_build", "bf16x_hip")
ARCH = "gfx950"

COMMON = ["-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function",
          "-I" + os.path.join(ROOT, "include")]
HIP_FLAGS = [f"--offload-arch={ARCH}", "-mcode-object-version=5",
             "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
             "-fno-gpu-rdc", "-munsafe-fp-atomics"]


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (ROCm is required to build the BF16X HIP library)")


def _compile(src: str, verbose: bool) -> str:
    obj = os.path.join(BUILD_DIR, os.path.basename(src) + ".o")
    cmd = [_hipcc()] + COMMON
    if src.endswith(".hip"):
        cmd += HIP_FLAGS + ["-x", "hip"]
    cmd += ["-c", src, "-o", obj]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    noise = ("packed-fp32-ops", "is not a recognized feature")
    msg = "\n".join(l for l in (r.stdout + r.stderr).splitlines() if not any(n in l for n in noise))
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{msg}")
    if msg.strip() and verbose:
        print(msg, flush=True)
    return obj


def _build_host(verbose: bool) -> None:
    """_host.so: links libbf16x_hip.so beside it and torch's libraries (which
    are loaded already when it is imported)."""
    import torch
    inc = os.path.join(os.path.dirname(torch.__file__), "include")
    tlib = os.path.join(os.path.dirname(torch.__file__), "lib")
    tmp = HOST_OUT + ".tmp"
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-DUSE_ROCM", "-D__HIP_PLATFORM_AMD__",
           "-I" + os.path.join(ROOT, "include"), "-isystem", inc, "-isystem",
           os.path.join(inc, "torch", "csrc", "api", "include"), "-isystem", sysconfig.get_paths()["include"],
           "-isystem", "/opt/rocm/include", HOST_SRC, "-o", tmp, "-L" + tlib, "-ltorch_python", "-ltorch_cpu",
           "-ltorch", "-lc10", "-lc10_hip", "-L" + HERE, "-lbf16x_hip", "-Wl,-rpath,$ORIGIN"]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("g++ failed on host_ext.cpp:\n" + r.stdout + r.stderr)
    os.replace(tmp, HOST_OUT)


def build(verbose: bool = False) -> str:
    os.makedirs(BUILD_DIR, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.cpp")))
    srcs.remove(HOST_SRC)
    with cf.ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        objs = list(ex.map(lambda s: _compile(s, verbose), srcs))
    tmp = OUT + ".tmp"
    cmd = [_hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp] + objs + \
        ["-Wl,-rpath,/opt/rocm/lib", "-lpthread"]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stdout + r.stderr)
    os.replace(tmp, OUT)
    _build_host(verbose)
    return OUT


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
