"""Build recipe of libgmdn_scan.so and libgmdn_ops.so, in-tree.

``python -m gmdn_amd.build`` (from the package root directory) or
``gmdn_amd.build.build()`` compiles every ``csrc/*.hip`` translation unit to
an object in parallel (hipcc for gfx950), links them into
``gmdn_amd/libgmdn_scan.so``, and builds the torch operators over it,
``csrc/torch_ops.cpp``, into ``gmdn_amd/libgmdn_ops.so`` (host code only).
"""
from __future__ import annotations

import concurrent.futures
import glob
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
PKG_ROOT = os.path.dirname(HERE)
CSRC = os.path.join(PKG_ROOT, "csrc")
OUT = os.path.join(HERE, "libgmdn_scan.so")
OPS_SRC = os.path.join(CSRC, "torch_ops.cpp")
OPS_OUT = os.path.join(HERE, "libgmdn_ops.so")
OBJ_DIR = os.path.join(PKG_ROOT, "_build")

ARCH = "gfx950"
HIPCC = os.environ.get("HIPCC", shutil.which("hipcc") or "/opt/rocm/bin/hipcc")

# Packed fp32 ops are disabled: hipcc -O3 forms v_pk_{add,mul,fma}_f32 on its
# own, and the library keeps to scalar fp32 VALU for the state arithmetic.
# MFMA results stay in arch VGPRs (no v_accvgpr moves before the VALU work
# on them: the scan kernels pack every product into the next operand).
COMMON_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-mllvm", "-amdgpu-mfma-vgpr-form=1",
    "-Wno-unused-command-line-argument",
]


def _compile(src: str, verbose: bool) -> str:
    obj = os.path.join(OBJ_DIR, os.path.basename(src) + ".o")
    cmd = [HIPCC, *COMMON_FLAGS, "-c", src, "-o", obj]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr}")
    return obj


def _run(cmd, what: str, verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{what} failed:\n{r.stderr}")


def _compile_ops(verbose: bool) -> str:
    """The torch operators' object (torch's headers and ABI; no device code)."""
    import torch
    obj = os.path.join(OBJ_DIR, "torch_ops.cpp.o")
    inc = os.path.join(os.path.dirname(torch.__file__), "include")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    _run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-isystem", inc, "-isystem",
          os.path.join(inc, "torch", "csrc", "api", "include"), "-isystem", os.path.join(rocm, "include"), "-c", OPS_SRC,
          "-o", obj], f"compiling {OPS_SRC}", verbose)
    return obj


def _link_ops(obj: str, verbose: bool) -> None:
    import torch
    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    tmp = OPS_OUT + ".tmp"
    _run([os.environ.get("CXX", "g++"), "-shared", obj, "-o", tmp, "-L", lib, "-ltorch", "-ltorch_cpu", "-lc10",
          "-lc10_hip", "-L", HERE, "-lgmdn_scan", "-Wl,-rpath,$ORIGIN"], "linking the torch operators", verbose)
    os.replace(tmp, OPS_OUT)


def build(verbose: bool = False, jobs: int | None = None) -> str:
    """Compile all HIP sources for gfx950 and link the C-ABI shared library,
    then the torch operators over it."""
    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    if not srcs:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    jobs = jobs or min(len(srcs), os.cpu_count() or 4, 8)
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as ex:
        ops_obj = ex.submit(_compile_ops, verbose)
        objs = list(ex.map(lambda s: _compile(s, verbose), srcs))
        ops_obj = ops_obj.result()
    tmp = OUT + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp]
    _run(cmd, "link", verbose)
    os.replace(tmp, OUT)
    _link_ops(ops_obj, verbose)
    return OUT


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
