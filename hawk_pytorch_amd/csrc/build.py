"""Builds libhawk_hip.so (the C-ABI HIP library) in-tree with hipcc for gfx950, and _hawk_torch.so (the host side of
eager calls, no device code) with g++ against the installed torch.

Usage:  python -m hawk_pytorch_amd.csrc.build [--force]
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

CSRC = os.path.dirname(os.path.abspath(__file__))
LIB_NAME = "libhawk_hip.so"
LIB_PATH = os.path.join(CSRC, LIB_NAME)
NATIVE_NAME = "_hawk_torch.so"
NATIVE_PATH = os.path.join(CSRC, NATIVE_NAME)
SOURCES = ["hawk_scan.hip", "hawk_conv.hip", "hawk_step.hip", "hawk_gates.hip", "hawk_block.hip", "hawk_decode.hip", "hawk_train.hip", "hawk_wgrad.hip", "hawk_probe.hip", "hawk_capi.hip"]
HEADERS = ["hawk_scan.h", "hawk_device.h", "hawk_reduce.h", "hawk_tile.h", os.path.join("..", "..", "include", "hawk_hip.h")]

# Packed-FP32 VALU instructions are switched off for all device code.
HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; libhawk_hip.so cannot be built")
    return exe


def _run(cmd):
    proc = subprocess.run(cmd, cwd=CSRC, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError("command failed: %s\n%s\n%s" % (" ".join(cmd), proc.stdout, proc.stderr))
    return proc


def build_native(force: bool = True, verbose: bool = False) -> str:
    """Compile the torch extension module.  Returns its path."""
    import sysconfig

    import torch

    source, header = os.path.join(CSRC, "hawk_torch.cpp"), os.path.join(CSRC, "..", "..", "include", "hawk_hip.h")
    if not force and os.path.exists(NATIVE_PATH) and os.path.getmtime(NATIVE_PATH) >= max(map(os.path.getmtime, (source, header))):
        return NATIVE_PATH
    if verbose:
        print("g++ hawk_torch.cpp", flush=True)
    root = os.path.dirname(torch.__file__)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    tmp = NATIVE_PATH + ".%d.tmp" % os.getpid()
    _run([shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Wno-unused-function",
          "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch.compiled_with_cxx11_abi(),
          "-isystem", os.path.join(root, "include"),
          "-isystem", os.path.join(root, "include", "torch", "csrc", "api", "include"),
          "-isystem", sysconfig.get_paths()["include"], "-isystem", os.path.join(rocm, "include"), source, "-o", tmp,
          "-L" + os.path.join(root, "lib"), "-lc10", "-lc10_hip", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-ltorch_python"])
    os.replace(tmp, NATIVE_PATH)
    return NATIVE_PATH


def build(force: bool = True, verbose: bool = False) -> str:
    """Compile every translation unit and link the shared library, and the torch extension beside it.  Returns the
    library's path."""
    hipcc = _hipcc()
    objdir = os.path.join(CSRC, "build")
    os.makedirs(objdir, exist_ok=True)
    newest_header = max(os.path.getmtime(os.path.join(CSRC, h)) for h in HEADERS)

    def compile_one(src):
        obj = os.path.join(objdir, src.replace(".hip", ".o"))
        src_path = os.path.join(CSRC, src)
        stale = (
            force
            or not os.path.exists(obj)
            or os.path.getmtime(obj) < max(os.path.getmtime(src_path), newest_header)
        )
        if stale:
            if verbose:
                print("hipcc", src, flush=True)
            _run([hipcc, *HIPCC_FLAGS, "-c", src_path, "-o", obj])
        return obj

    with ThreadPoolExecutor(max_workers=len(SOURCES) + 1) as pool:
        native = pool.submit(build_native, force, verbose)
        objs = list(pool.map(compile_one, SOURCES))
        native.result()
    _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB_PATH, *objs])
    return LIB_PATH


if __name__ == "__main__":
    path = build(force="--force" in sys.argv, verbose=True)
    print(path)
