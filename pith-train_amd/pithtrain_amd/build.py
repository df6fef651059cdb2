"""Builds libpith_hip.so (the C-ABI library of HIP kernels) for gfx950 with hipcc, and _pith_torch.so (the operators' native
host path on top of it) with the host compiler.

Both are placed in-tree under pithtrain_amd/lib/ so that they travel with a
source snapshot; nothing is installed into site-packages and nothing is compiled at import time.
Run as `python -m pithtrain_amd.build` (from the pith-train_amd/ directory) or call build().
"""

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
SRC_DIR = os.path.join(os.path.dirname(PKG_DIR), "csrc")
INCLUDE_DIR = os.path.join(os.path.dirname(os.path.dirname(PKG_DIR)), "include")
LIB_DIR = os.path.join(PKG_DIR, "lib")
LIB_PATH = os.path.join(LIB_DIR, "libpith_hip.so")
OBJ_DIR = os.path.join(LIB_DIR, "obj")
EXT_SRC = os.path.join(SRC_DIR, "host", "torch_ops.cpp")
EXT_PATH = os.path.join(LIB_DIR, "_pith_torch.so")

SOURCES = ["api.hip", "combine.hip", "norm_rope.hip", "mla_assemble.hip", "attn_fwd.hip", "attn_fwd_direct.hip", "attn_fwd_duo.hip", "attn_bwd_dq.hip", "attn_bwd_dq_direct.hip", "attn_bwd_dq_duo.hip", "attn_bwd_dq_ds.hip", "attn_bwd_dkdv.hip", "attn_bwd_pair.hip", "attn_bwd_chunks.hip", "attn_bwd_dkdv_d64.hip", "attn_bwd_dkdv_d128.hip", "attn_bwd_dkdv_wide.hip", "attn_bwd_dkdv_d192.hip"]

# -packed-fp32-ops is switched off on purpose: some packed fp32 forms have produced wrong results
# on the target machines. Code object v5 is understood by both the ROCm 7.0 runtime bundled with
# PyTorch and the system ROCm 7.2 runtime.
HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-mcode-object-version=5",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
]

# Backward over several chunks: a share of few workgroups is as long as its longest walk, one wave to a SIMD, which fetches its loop anew at every
# turn. Three scalar instructions in front of it (tiles_of_wave) moved it off the fetch lines; forward + backward of 64 features, us, before
# them / after / with loops on 64 bytes: 2146 x 4 heads, 8 ranks, rank 3 358 / 368 / 356, 848 x 16, rank 0 221 / 225 / 220, 3 x 1856 x 4, rank 6
# contiguous 401 / 410 / 401; 95 such shares 0.7 % faster, 205 of 128 and 192 features equal. Not the forward (all files aligned: 2884 x 8/2 of 128
# without a mask 43.8 / 47.8).
SOURCE_FLAGS = {"attn_bwd_chunks.hip": ["-falign-loops=64"]}


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; libpith_hip.so can only be built with the ROCm toolchain")
    return exe


def _compile(src: str, extra: list) -> str:
    obj = os.path.join(OBJ_DIR, os.path.splitext(src)[0] + ".o")
    cmd = [_hipcc(), *HIPCC_FLAGS, *SOURCE_FLAGS.get(src, []), *extra, "-I", INCLUDE_DIR, "-I", SRC_DIR, "-c", os.path.join(SRC_DIR, src), "-o", obj]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(line for line in proc.stderr.splitlines() if noise not in line)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _compile_ext() -> str:
    """Object file of the native host path: plain host code against the installed PyTorch's headers."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths

    obj = os.path.join(OBJ_DIR, "torch_ops.o")
    includes = [INCLUDE_DIR, *include_paths(), sysconfig.get_paths()["include"], "/opt/rocm/include"]
    cmd = [shutil.which("g++") or "c++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           "-DTORCH_API_INCLUDE_EXTENSION_H", "-DTORCH_EXTENSION_NAME=_pith_torch",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *[a for p in includes for a in ("-isystem" if p != INCLUDE_DIR else "-I", p)], "-c", EXT_SRC, "-o", obj]  # fmt: skip
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"the host compiler failed on {EXT_SRC}:\n{proc.stderr}")
    return obj


def _link_ext(obj: str) -> None:
    """Torch's libraries are in the process before this one is loaded, so they need no rpath; libpith_hip.so is beside it."""
    from torch.utils.cpp_extension import library_paths

    libs = [a for p in library_paths() for a in ("-L", p)]
    cmd = [shutil.which("g++") or "c++", "-shared", obj, "-o", EXT_PATH, *libs, "-lc10", "-ltorch_cpu", "-ltorch", "-lc10_hip", "-ltorch_hip",
           "-ltorch_python", "-L", LIB_DIR, "-l:libpith_hip.so", "-Wl,-rpath,$ORIGIN"]  # fmt: skip
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link of {EXT_PATH} failed:\n{proc.stderr}")


def build(verbose: bool = True, extra_flags=()) -> str:
    """Compiles every HIP source and links libpith_hip.so, then the native host path. Returns the library path."""
    os.makedirs(OBJ_DIR, exist_ok=True)
    with ThreadPoolExecutor(max_workers=min(8, len(SOURCES))) as pool:
        ext = pool.submit(_compile_ext)
        objs = list(pool.map(lambda s: _compile(s, list(extra_flags)), SOURCES))
        ext_obj = ext.result()
    # libamdhip64 is referenced by soname only (no rpath): inside a PyTorch process the loader
    # then resolves it to the HIP runtime PyTorch has already loaded instead of a second copy.
    cmd = [_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-mcode-object-version=5", *objs, "-o", LIB_PATH]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed:\n{proc.stderr}")
    _link_ext(ext_obj)
    if verbose:
        for path in (LIB_PATH, EXT_PATH):
            print(f"built {path} ({os.path.getsize(path)} bytes)")
    return LIB_PATH


if __name__ == "__main__":
    build(extra_flags=sys.argv[1:])
