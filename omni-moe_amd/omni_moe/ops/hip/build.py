"""Builds libomni_moe_hip.so (gfx950) and, on top of it, the torch host path _native.so, in-tree with hipcc.

Run as ``python -m omni_moe.ops.hip.build`` (with ``omni-moe_amd`` on sys.path) or
call :func:`build_library`.  No GPU is needed to compile.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
PKG_ROOT = os.path.abspath(os.path.join(HERE, "..", "..", ".."))          # omni-moe_amd/
REPO_ROOT = os.path.abspath(os.path.join(PKG_ROOT, ".."))
CSRC = os.path.join(PKG_ROOT, "csrc")
INCLUDE = os.path.join(REPO_ROOT, "include")
LIB_PATH = os.path.join(HERE, "libomni_moe_hip.so")
NATIVE_PATH = os.path.join(HERE, "_native.so")
OBJ_DIR = os.path.join(PKG_ROOT, "build")

SOURCES = ["gemm.hip", "gemm_tiles.hip", "gemm_tiles_bf16.hip", "gemm_tiles_f16.hip", "router.hip", "expert.hip", "backward.hip", "schedule.hip", "layer.hip", "few_tokens.hip", "mlp_bwd.hip", "api.hip"]

# packed-fp32 VALU forms are switched off for all device code of this library
HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", INCLUDE, "-I", CSRC, "-Wno-unused-value",
]


def _hipcc() -> str:
    for c in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if c and (os.path.isabs(c) and os.path.exists(c) or not os.path.isabs(c)):
            return c
    raise RuntimeError("hipcc not found")


def _compile(src: str, verbose: bool) -> str:
    obj = os.path.join(OBJ_DIR, os.path.splitext(src)[0] + ".o")
    cmd = [_hipcc(), *HIPCC_FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{r.stdout}\n{r.stderr}")
    if verbose and r.stderr.strip():
        print(r.stderr, file=sys.stderr)
    return obj


def _run(cmd, verbose: bool, what: str) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{what} failed:\n{r.stdout}\n{r.stderr}")


def _compile_native(verbose: bool) -> str:
    """The host path for torch: host code only, against torch's headers."""
    import sysconfig

    from torch.utils import cpp_extension
    obj = os.path.join(OBJ_DIR, "torch_ops.o")
    includes = [a for p in [INCLUDE, *cpp_extension.include_paths("cuda"), sysconfig.get_paths()["include"]] for a in ("-I", p)]
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_EXTENSION_NAME=_native",
          "-DTORCH_API_INCLUDE_EXTENSION_H", *includes, "-c", os.path.join(CSRC, "torch_ops.cpp"), "-o", obj], verbose, "compiling torch_ops.cpp")
    return obj


def _link_native(obj: str, verbose: bool) -> str:
    from torch.utils import cpp_extension
    torch_lib = cpp_extension.library_paths("cuda")[0]
    _run(["g++", "-shared", "-fPIC", obj, "-L", HERE, "-lomni_moe_hip", "-L", torch_lib, "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python",
          "-Wl,-rpath,$ORIGIN", "-o", NATIVE_PATH], verbose, "linking _native.so")
    return NATIVE_PATH


def build_library(verbose: bool = False, jobs: int = 8) -> str:
    os.makedirs(OBJ_DIR, exist_ok=True)
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        native = ex.submit(_compile_native, verbose)
        objs = list(ex.map(lambda s: _compile(s, verbose), SOURCES))
        native_obj = native.result()
    _run([_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", LIB_PATH], verbose, "linking libomni_moe_hip.so")
    _link_native(native_obj, verbose)
    return LIB_PATH


if __name__ == "__main__":
    print(build_library(verbose=True))
