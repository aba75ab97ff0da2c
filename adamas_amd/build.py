"""Builds libadamas_hip.so (hand-written HIP kernels + the C ABI) for gfx950 with hipcc, and adamas_host.so (the native
host side of the operators of a decode token) with g++.

The library is built in-tree (adamas_amd/lib/) so that it travels with the source tree; nothing is
installed into site-packages and nothing is compiled at import time.
"""
from __future__ import annotations

import os
import shutil
import subprocess
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC_DIR = PKG_DIR / "csrc"
LIB_DIR = PKG_DIR / "lib"
LIB_PATH = LIB_DIR / "libadamas_hip.so"
HOST_PATH = LIB_DIR / "adamas_host.so"

SOURCES = ["hadamard.hip", "estimate.hip", "topk.hip", "attention.hip", "fused_step.hip",
           "prefill.hip", "decoder_ops.hip"]

HIPCC_FLAGS = [
    "-O3",
    "--offload-arch=gfx950",
    "-std=c++17",
    "-fPIC",
    # packed fp32 instructions are switched off for all device code of this library
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # the first 14 registers of kernel arguments arrive with the workgroup instead of being fetched by
    # it: a memory round trip off the start of every kernel whose first addresses come from them (the
    # kernels of the decode step list those first).  One layer of a step without / with it, in us:
    # 4096 tokens 12.9 / 12.3, 32768 19.2 / 18.5, 131072 40.6 / 39.8, 23989 at 32:8 heads, budget 1024
    # 22.2 / 21.8, 16 sequences of 8192 to 32768 82.5 / 81.6.
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
]


def find_hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found: set HIPCC or put /opt/rocm/bin on PATH")


def _run(cmd, verbose):
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if verbose or proc.returncode != 0:
        print(" ".join(cmd))
        print(proc.stdout)
        print(proc.stderr)
    if proc.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed with exit code {proc.returncode}")


def build_library(verbose: bool = False, jobs: int = 0) -> Path:
    """Compile every HIP source (one hipcc process each, side by side) and link them into
    adamas_amd/lib/libadamas_hip.so; returns its path.  Every call recompiles everything."""
    from concurrent.futures import ThreadPoolExecutor

    LIB_DIR.mkdir(parents=True, exist_ok=True)
    obj_dir = LIB_DIR / "obj"
    obj_dir.mkdir(exist_ok=True)
    hipcc = find_hipcc()
    jobs = jobs or min(len(SOURCES), os.cpu_count() or 1, 8)
    objects = [obj_dir / (Path(src).stem + ".o") for src in SOURCES]
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        list(pool.map(lambda so: _run([hipcc, *HIPCC_FLAGS, "-c", str(CSRC_DIR / so[0]), "-o",
                                       str(so[1])], verbose), zip(SOURCES, objects)))
    _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *[str(o) for o in objects], "-o",
          str(LIB_PATH)], verbose)
    _run(host_command(), verbose)
    return LIB_PATH


def host_command() -> list:
    """g++ for the extension module of csrc/host_ops.cpp: no device code, torch's headers and libraries (which the
    process has loaded by the time the module is), the HIP library beside it."""
    import sysconfig

    import torch

    root = Path(torch.__file__).resolve().parent
    rocm = Path(find_hipcc()).resolve().parents[1]
    includes = [root / "include", root / "include" / "torch" / "csrc" / "api" / "include", rocm / "include",
                sysconfig.get_paths()["include"]]
    return ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
            f'-DADAMAS_TORCH_VERSION="{torch.__version__}"',
            *[f"-I{d}" for d in includes], str(CSRC_DIR / "host_ops.cpp"), "-o", str(HOST_PATH),
            f"-L{root / 'lib'}", "-ltorch_python", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip",
            f"-L{LIB_DIR}", f"-l:{LIB_PATH.name}", "-Wl,-rpath,$ORIGIN"]


if __name__ == "__main__":
    print(build_library(verbose=True))
