"""Builds libtdb_attn.so (HIP kernels + C ABI, hipcc for gfx950) and _host.so (the operators' native front, host code
only), in-tree."""
from __future__ import annotations

import os
import shutil
import subprocess
import sysconfig
from concurrent.futures import ThreadPoolExecutor

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
LIB_PATH = os.path.join(PKG, "libtdb_attn.so")
HOST_PATH = os.path.join(PKG, "_host.so")
SOURCES = ("capi.hip", "attn_generic.hip", "attn_f32.hip", "attn_f32_split.hip", "attn_short.hip", "encoder.hip", "gemm.hip", "attn_mfma.hip", "attn_resident.hip")

# packed-fp32 VALU forms are switched off for every device compile
HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-mllvm", "-amdgpu-mfma-vgpr-form=1",      # MFMA accumulators in VGPRs: no accvgpr copies around the softmax
    "-Wno-unused-command-line-argument",
    "-I", os.path.join(ROOT, "include"), "-I", CSRC,
]


def hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; libtdb_attn.so cannot be built")
    return exe


def _compile(src: str, obj_dir: str) -> str:
    obj = os.path.join(obj_dir, os.path.splitext(src)[0] + ".o")
    cmd = [hipcc(), *HIPCC_FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{res.stderr[-4000:]}")
    return obj


def _compile_host() -> str:
    """The CPython module over the C ABI: plain C++ against PyTorch's headers, no device code."""
    import torch
    from torch.utils.cpp_extension import include_paths
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(hipcc())))
    tmp = HOST_PATH + ".tmp"
    cmd = [shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wno-attributes",
           "-D__HIP_PLATFORM_AMD__=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *(f for d in include_paths() + [sysconfig.get_paths()["include"]] for f in ("-isystem", d)),
           "-isystem", os.path.join(rocm, "include"), "-I", os.path.join(ROOT, "include"), "-I", CSRC,
           *(os.path.join(CSRC, f) for f in ("host.cpp", "host_encoder.cpp")), "-o", tmp, "-L", os.path.join(os.path.dirname(torch.__file__), "lib"),
           "-ltorch_python", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed on the host module:\n{res.stderr[-4000:]}")
    os.replace(tmp, HOST_PATH)
    return HOST_PATH


def build_library(verbose: bool = False) -> str:
    """Compile every source and link the shared library.  Always recompiles."""
    obj_dir = os.path.join(PKG, "build")
    os.makedirs(obj_dir, exist_ok=True)
    with ThreadPoolExecutor(max_workers=len(SOURCES) + 1) as ex:
        host = ex.submit(_compile_host)
        objs = list(ex.map(lambda s: _compile(s, obj_dir), SOURCES))
    tmp = LIB_PATH + ".tmp"
    cmd = [hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", tmp]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr[-4000:]}")
    os.replace(tmp, LIB_PATH)
    host.result()
    if verbose:
        print("built", LIB_PATH, HOST_PATH)
    return LIB_PATH


if __name__ == "__main__":
    build_library(verbose=True)
