"""In-tree build of the C-ABI runtime library ``liboeq_hip.so`` with hipcc and of the torch operators' autograd kernels
``liboeq_torch.so`` (host code only) with the C++ compiler.

``python -m openequivariance_amd.build_ext`` (or ``__graft_entry__.build()``)
compiles ``csrc/oeq_hip.cpp`` for gfx950 and ``csrc/oeq_torch.cpp`` against the installed torch and leaves the shared
objects next to the sources, where :mod:`openequivariance_amd.runtime` and :mod:`openequivariance_amd.autograd_glue` load
them from.  The libraries are never built implicitly at import time.
"""
from __future__ import annotations

import os
import pathlib
import shutil
import subprocess
import sys

PKG_DIR = pathlib.Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
LIB_PATH = CSRC / "liboeq_hip.so"
TORCH_LIB_PATH = CSRC / "liboeq_torch.so"
ROCM = pathlib.Path(os.environ.get("ROCM_PATH", "/opt/rocm"))

# -packed-fp32-ops is switched off for every device compilation of this project
PACKED_FP32_OFF = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def hipcc_path() -> str:
    cand = shutil.which("hipcc") or str(ROCM / "bin" / "hipcc")
    if not os.path.exists(cand):
        raise RuntimeError("hipcc not found; set ROCM_PATH")
    return cand


def build_native(verbose: bool = True) -> pathlib.Path:
    cmd = [hipcc_path(), "--offload-arch=gfx950", "-O2", "-std=c++17", "-fPIC", "-shared",
           *PACKED_FP32_OFF,
           str(CSRC / "oeq_hip.cpp"), "-o", str(LIB_PATH),
           f"-L{ROCM / 'lib'}", "-lhiprtc", f"-Wl,-rpath,{ROCM / 'lib'}", "-Wl,--enable-new-dtags"]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed:\n{res.stdout}\n{res.stderr}")
    if verbose and res.stderr.strip():
        print(res.stderr, file=sys.stderr)
    build_torch_ops(verbose)
    return LIB_PATH


def build_torch_ops(verbose: bool = True) -> pathlib.Path:
    import torch
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        raise RuntimeError("no C++ compiler found (g++ or c++)")
    root = pathlib.Path(torch.__file__).resolve().parent
    cmd = [cxx, "-O2", "-std=c++17", "-fPIC", "-shared", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f"-I{root / 'include'}", f"-I{root / 'include' / 'torch' / 'csrc' / 'api' / 'include'}",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM", f"-I{ROCM / 'include'}",
           str(CSRC / "oeq_torch.cpp"), "-o", str(TORCH_LIB_PATH), f"-L{root / 'lib'}", "-ltorch", "-ltorch_cpu", "-lc10",
           "-lc10_hip", "-lamdhip64"]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{cxx} failed:\n{res.stdout}\n{res.stderr}")
    return TORCH_LIB_PATH


if __name__ == "__main__":
    print(build_native())
