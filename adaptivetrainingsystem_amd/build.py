"""Builds libats_gfx950.so (hand-written HIP kernels + C ABI) with hipcc for gfx950, and _ats_torch.so (the host side of
its shortest calls) with the C++ compiler.

The library is built in-tree (adaptivetrainingsystem_amd/lib/) so that it travels
with the source tree; nothing is compiled at import time.
Run ``python -m adaptivetrainingsystem_amd.build`` or call ``build_library()``.
"""
from __future__ import annotations

import glob
import os
import shutil
import subprocess
import sys
import tempfile

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
CSRC_DIR = os.path.join(PKG_DIR, "csrc")
LIB_DIR = os.path.join(PKG_DIR, "lib")
LIB_PATH = os.path.join(LIB_DIR, "libats_gfx950.so")
BINDING_PATH = os.path.join(LIB_DIR, "_ats_torch.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def find_hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (set HIPCC or add /opt/rocm/bin to PATH)")


def sources():
    return sorted(glob.glob(os.path.join(CSRC_DIR, "*.hip")))


def _compile_binding(obj: str):
    """Starts the compilation of the host side of the short calls (csrc/torch_binding.cpp), plain C++ against torch's headers."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths
    cxx = os.environ.get("CXX") or shutil.which("g++") or shutil.which("c++")
    if not cxx:
        raise RuntimeError("no C++ compiler found (set CXX)")
    # (the first two are what the HIP headers ask of a compiler that is not hipcc)
    cmd = [cxx, "-O2", "-std=c++17", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-DTORCH_API_INCLUDE_EXTENSION_H",
           "-DTORCH_EXTENSION_NAME=_ats_torch", *("-I" + d for d in include_paths(device_type="cuda")),
           "-I" + sysconfig.get_paths()["include"], "-c", os.path.join(CSRC_DIR, "torch_binding.cpp"), "-o", obj]
    link = [cxx, "-shared", obj, "-L" + os.path.join(os.path.dirname(torch.__file__), "lib"), "-lc10", "-lc10_hip", "-ltorch_cpu",
            "-ltorch", "-ltorch_python", "-L" + LIB_DIR, "-l:libats_gfx950.so", "-Wl,-rpath,$ORIGIN"]
    return cmd, link


def build_library(verbose: bool = True, jobs: int = 6) -> str:
    """Compiles every .hip source to an object (in parallel) and links the shared library."""
    hipcc = find_hipcc()
    os.makedirs(LIB_DIR, exist_ok=True)
    obj_dir = os.path.join(LIB_DIR, "obj")
    os.makedirs(obj_dir, exist_ok=True)
    compile_flags = [f for f in HIPCC_FLAGS if f != "-shared"]
    procs, objs = [], []

    def start(cmd):     # (output to a file: a compiler with much to say would wait for a reader of its pipe, and this waits for it)
        log = tempfile.TemporaryFile("w+", errors="replace")
        return subprocess.Popen(cmd, stdout=log, stderr=subprocess.STDOUT), log

    binding_obj = os.path.join(obj_dir, "torch_binding.o")
    binding_cmd, binding_link = _compile_binding(binding_obj)
    procs.append(("torch_binding.cpp", *start(binding_cmd)))
    for src in sources():
        obj = os.path.join(obj_dir, os.path.basename(src)[:-4] + ".o")
        objs.append(obj)
        cmd = [hipcc, *compile_flags, "-c", src, "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((src, *start(cmd)))
        while sum(p.poll() is None for _, p, _ in procs) >= jobs:
            for _, p, _ in procs:
                if p.poll() is None:
                    p.wait()
                    break
    failed = False
    for src, p, log in procs:
        p.wait()
        log.seek(0)
        out = "\n".join(l for l in log.read().splitlines() if "packed-fp32-ops" not in l)
        if p.returncode != 0:
            failed = True
            print(f"FAILED: {src}\n{out}", file=sys.stderr)
        elif verbose and out.strip():
            print(out)
    if failed:
        raise RuntimeError("hipcc failed")
    tmp = LIB_PATH + ".tmp"
    cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", tmp]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    os.replace(tmp, LIB_PATH)
    tmp = BINDING_PATH + ".tmp"
    subprocess.check_call([*binding_link, "-o", tmp])
    os.replace(tmp, BINDING_PATH)
    return LIB_PATH


if __name__ == "__main__":
    print(build_library())
