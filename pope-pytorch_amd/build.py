"""Build libpope_hip.so and _pope_host.so in-tree (hipcc for gfx950, g++ for the host module; no cmake).

    python pope-pytorch_amd/build.py [-j N]

Each source in csrc/ is compiled to an object under _build/ (parallel), then
linked into pope_amd/libpope_hip.so; csrc_torch/pope_host.cpp (torch's C++ API, no device
code) becomes the Python module pope_amd/_pope_host.so, linked against it.  Always rebuilds.
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT_DIR = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "pope_amd", "libpope_hip.so")
HOST_SRC = os.path.join(HERE, "csrc_torch", "pope_host.cpp")
HOST_LIB = os.path.join(HERE, "pope_amd", "_pope_host.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

FLAGS = [
    "-O3", "-std=c++17", "-fPIC", "--offload-arch=gfx950",
    # packed fp32 VALU ops are kept out of every kernel
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-munsafe-fp-atomics",
    "-Wno-unused-result",
]


def sources():
    return sorted(f for f in os.listdir(CSRC) if f.endswith((".hip", ".cpp")))


def compile_one(src: str) -> str:
    obj = os.path.join(OUT_DIR, src + ".o")
    cmd = [HIPCC, *FLAGS, "-I", CSRC, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed: {src}\n{err}")
    return obj


def compile_host() -> str:
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths
    rocm = os.path.dirname(os.path.dirname(HIPCC))
    obj = os.path.join(OUT_DIR, "pope_host.o")
    inc = [*include_paths(), sysconfig.get_paths()["include"], os.path.join(rocm, "include")]
    # the HIP headers' own platform macros, as hipcc sets them
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-DTORCH_EXTENSION_NAME=_pope_host",
           "-DTORCH_API_INCLUDE_EXTENSION_H", *(f"-isystem{d}" for d in inc), "-c", HOST_SRC, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed: {HOST_SRC}\n{r.stderr}")
    return obj


def link_host(obj: str) -> str:
    import torch
    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    tmp = HOST_LIB + ".tmp"
    cmd = ["g++", "-shared", "-o", tmp, obj, "-L", os.path.dirname(LIB), "-l:libpope_hip.so", "-L", lib, "-ltorch",
           "-ltorch_cpu", "-ltorch_python", "-lc10", "-lc10_hip", "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed\n" + r.stderr)
    os.replace(tmp, HOST_LIB)
    return HOST_LIB


def build(jobs: int = 8) -> str:
    os.makedirs(OUT_DIR, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        host = ex.submit(compile_host)
        objs = list(ex.map(compile_one, sources()))
        host_obj = host.result()
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed\n" + r.stderr)
    os.replace(tmp, LIB)
    link_host(host_obj)
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("-j", type=int, default=min(8, os.cpu_count() or 1))
    a = ap.parse_args()
    print(build(a.j))
