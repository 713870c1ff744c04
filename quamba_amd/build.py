"""Builds libquamba_amd.so (HIP, gfx950) in-tree with hipcc.

Usage: python -m quamba_amd.build [--force]
The library is cross-compiled without a GPU; the built file sits beside this module so that it
travels with the source tree.  Beside it goes _host.so, the host side of the mixers' calls (C++ against torch's
headers, no device code).
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "csrc", "build")
LIB = os.path.join(HERE, "libquamba_amd.so")
HOST = os.path.join(HERE, "_host.so")
HOST_SRC = os.path.join(HERE, "host", "layer_call.cpp")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

# -ffp-contract=off: every fused multiply-add in the kernels is written explicitly, so the
# arithmetic order is the one in the source.  Packed-fp32 instructions are disabled.
FLAGS = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unknown-warning-option", "-Wno-pass-failed",
]


def sources():
    return sorted(f for f in os.listdir(CSRC) if f.endswith(".hip"))


def _newer(a, b):
    return (not os.path.exists(b)) or os.path.getmtime(a) > os.path.getmtime(b)


def _compile(src, force):
    obj = os.path.join(BUILD, src[:-4] + ".o")
    path = os.path.join(CSRC, src)
    deps = [path, os.path.join(CSRC, "qa_common.hpp"), os.path.join(HERE, "..", "include", "quamba_amd.h")]
    deps += [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hpp")]
    if force or any(_newer(d, obj) for d in deps):
        cmd = [HIPCC, *FLAGS, "-c", path, "-o", obj]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"hipcc failed for {src}:\n{r.stdout}\n{r.stderr}")
        warn = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l and l.strip())
        if warn:
            sys.stderr.write(warn + "\n")
    return obj


def build_host(force=False):
    header = os.path.join(HERE, "..", "include", "quamba_amd.h")
    if not force and not any(_newer(d, HOST) for d in (HOST_SRC, header)):
        return
    import sysconfig

    import torch
    from torch.utils import cpp_extension
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f"-I{sysconfig.get_paths()['include']}", *(f"-I{d}" for d in cpp_extension.include_paths()), HOST_SRC, "-o", HOST,
           *(f"-L{d}" for d in cpp_extension.library_paths()), "-lc10", "-ltorch_cpu", "-ltorch_python"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compilation of {HOST_SRC} failed:\n{r.stdout}\n{r.stderr}")


def build(force=False, jobs=None):
    os.makedirs(BUILD, exist_ok=True)
    srcs = sources()
    jobs = jobs or min(len(srcs), int(os.environ.get("MAX_JOBS", "8")))
    with ThreadPoolExecutor(max_workers=max(1, jobs)) as ex:
        host = ex.submit(build_host, force)
        objs = list(ex.map(lambda s: _compile(s, force), srcs))
        host.result()
    if force or any(_newer(o, LIB) for o in objs):
        cmd = [HIPCC, "-shared", "-fPIC", f"--offload-arch={ARCH}", *objs, "-o", LIB]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    return LIB


if __name__ == "__main__":
    print(build(force="--force" in sys.argv))
