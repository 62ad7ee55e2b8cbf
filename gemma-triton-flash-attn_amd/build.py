"""Build libgfa.so (the gfx950 HIP kernels + C ABI) and _gfa_torch.so (the native host path of the
PyTorch entry points) in-tree, with hipcc and the host C++ compiler.

Usage: python gemma-triton-flash-attn_amd/build.py [--jobs N] [--verbose]

Every HIP translation unit is compiled for gfx950 only, with packed-fp32 VALU ops
disabled (``-target-feature -packed-fp32-ops``). Objects go to ``_build/``; the shared
library lands next to this file so it travels with the source tree.
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import importlib.util
import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libgfa.so")
TORCH_LIB = os.path.join(HERE, "_gfa_torch.so")
SOURCES = ["gfa_fwd.hip", "gfa_fwd_rows.hip", "gfa_bwd_dq.hip", "gfa_bwd_dkv.hip", "gfa_bwd_ds.hip", "gfa_segments.hip",
           "gfa_api.hip"]
ARCH = "gfx950"


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(path):
        raise RuntimeError("hipcc not found; install ROCm or put hipcc on PATH")
    return path


def common_flags() -> list[str]:
    return [
        f"--offload-arch={ARCH}",
        "-O3",
        "-std=c++17",
        "-fPIC",
        "-Wall",
        "-Wno-unused-function",
        # Keep hipcc from forming v_pk_{add,mul,fma}_f32 from scalar float code.
        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
        f"-I{os.path.join(HERE, '..', 'include')}",
    ]


def _compile(src: str, verbose: bool) -> str:
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    cmd = [hipcc(), *common_flags(), "-c", os.path.join(CSRC, src), "-o", obj]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in (res.stderr or "").splitlines() if noise not in l)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{err}")
    if verbose and err.strip():
        print(err)
    return obj


def build_torch(verbose: bool = False) -> str:
    """Compile and link _gfa_torch.so (host code only) against the installed PyTorch."""
    torch_dir = os.path.dirname(importlib.util.find_spec("torch").origin)
    inc = os.path.join(torch_dir, "include")
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(hipcc())))
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        raise RuntimeError("no host C++ compiler (g++) on PATH")
    tmp = TORCH_LIB + ".tmp"
    cmd = [cxx, "-O2", "-std=c++17", "-fPIC", "-shared", "-DTORCH_EXTENSION_NAME=_gfa_torch",
           "-DTORCH_API_INCLUDE_EXTENSION_H", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-I{os.path.join(HERE, '..', 'include')}", "-isystem", inc,
           "-isystem", os.path.join(inc, "torch", "csrc", "api", "include"),
           "-isystem", sysconfig.get_paths()["include"], "-isystem", os.path.join(rocm, "include"),
           os.path.join(CSRC, "gfa_torch.cpp"), "-o", tmp, f"-L{os.path.join(torch_dir, 'lib')}",
           "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip", "-ltorch_python"]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{cxx} failed on gfa_torch.cpp:\n{res.stderr}")
    os.replace(tmp, TORCH_LIB)
    return TORCH_LIB


def build(jobs: int = 4, verbose: bool = False) -> str:
    """Compile every HIP source and link libgfa.so, and build _gfa_torch.so beside it. Returns the
    path of libgfa.so."""
    os.makedirs(BUILD, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=max(1, jobs)) as ex:
        ext = ex.submit(build_torch, verbose)
        objs = list(ex.map(lambda s: _compile(s, verbose), SOURCES))
        ext.result()
    tmp = LIB + ".tmp"
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    os.replace(tmp, LIB)
    return LIB


def main(argv: list[str] | None = None) -> int:
    ap = argparse.ArgumentParser(description=__doc__)
    ap.add_argument("--jobs", type=int, default=4)
    ap.add_argument("--verbose", action="store_true")
    args = ap.parse_args(argv)
    print(build(args.jobs, args.verbose))
    return 0


if __name__ == "__main__":
    sys.exit(main())
