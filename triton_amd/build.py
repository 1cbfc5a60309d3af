"""Builds `libtriton_amd.so` (gfx950 code objects + the C ABI) in-tree with hipcc, and `_host.so` (the native half of the
host path, a CPython extension on torch's C++ API) with the host compiler.

Usage: `python -m triton_amd.build` (or `__graft_entry__.build()`).  hipcc cross-compiles for gfx950
on a machine without a GPU; the shared libraries land next to this file and are what `_native.py` loads.
"""
from __future__ import annotations

import concurrent.futures
import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
LIB = os.path.join(HERE, "libtriton_amd.so")
HOST_SRC = os.path.join(CSRC, "host_path.cpp")
HOST_LIB = os.path.join(HERE, "_host.so")

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

# -packed-fp32-ops is switched off for every translation unit of this library.
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def sources():
    return sorted(f for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(src: str, force: bool) -> str:
    obj = os.path.join(OBJ, src[:-4] + ".o")
    src_path = os.path.join(CSRC, src)
    if not force and os.path.exists(obj):
        deps = [src_path] + [os.path.join(CSRC, h) for h in os.listdir(CSRC) if h.endswith(".h")]
        deps.append(os.path.join(HERE, "..", "include", "triton_amd.h"))
        if all(os.path.getmtime(d) <= os.path.getmtime(obj) for d in deps):
            return obj
    cmd = [HIPCC, *FLAGS, "-c", src_path, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stdout}\n{r.stderr}")
    warn = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l and l.strip())
    if "warning" in warn:
        sys.stderr.write(warn + "\n")
    return obj


def _build_host(force: bool) -> None:
    deps = [HOST_SRC, os.path.join(CSRC, "gemm_limits.h"), os.path.join(CSRC, "mx_tiles.h"), os.path.join(HERE, "..", "include", "triton_amd.h")]
    if not force and os.path.exists(HOST_LIB) and all(os.path.getmtime(d) <= os.path.getmtime(HOST_LIB) for d in deps):
        return
    import torch
    base = os.path.dirname(os.path.abspath(torch.__file__))
    inc, lib = os.path.join(base, "include"), os.path.join(base, "lib")
    tmp = HOST_LIB + ".tmp"
    # (torch's own libraries are found by name: the extension is imported by a process that has imported torch)
    cmd = [os.environ.get("CXX") or shutil.which("g++") or "g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-Wall", f"-I{inc}",
           f"-I{os.path.join(inc, 'torch', 'csrc', 'api', 'include')}", f"-I{sysconfig.get_paths()['include']}",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", HOST_SRC, "-o", tmp, f"-L{lib}", "-lc10",
           "-ltorch_cpu", "-ltorch", "-ltorch_python"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed for {os.path.basename(HOST_SRC)}:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, HOST_LIB)


def build(force: bool = True, jobs: int = 8) -> str:
    os.makedirs(OBJ, exist_ok=True)
    srcs = sources()
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(jobs, len(srcs))) as ex:
        host = ex.submit(_build_host, force)
        objs = list(ex.map(lambda s: _compile(s, force), srcs))
        host.result()
    tmp = LIB + ".tmp"
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", tmp], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(force="--incremental" not in sys.argv))
