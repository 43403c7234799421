"""Ahead-of-time build of the gfx950 kernel library (``libsvdq_mi355x.so``) with hipcc, and of the host extension
(``_host.so``: the operators' checks in native code, on torch's C++ interface) with the host compiler.

Run as ``python -m nunchaku_rocm_amd.build``.  Both are built in-tree next to this file so that they travel
with the source tree; nothing is compiled at import time or at run time.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libsvdq_mi355x.so")
HOST = os.path.join(HERE, "_host.so")
SOURCES = ["common.hip", "quantize.hip", "gemm_w4a4.hip", "gemm_w4a4_split.hip", "gemm_w4a4_wide.hip", "awq_gemv.hip", "awq_gemm.hip", "attention.hip", "layout.hip"]
FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # packed fp32 VALU ops stay off: plain v_fma_f32 / v_mul_f32 only
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]  # fmt: skip


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (set HIPCC or add /opt/rocm/bin to PATH)")


def host_command(out: str) -> list[str]:
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths, library_paths

    flags = [f"-I{p}" for p in (*include_paths(), sysconfig.get_paths()["include"])] + [f"-L{p}" for p in library_paths()]
    compiler = os.environ.get("CXX") or shutil.which("g++") or os.path.join(os.path.dirname(os.path.realpath(hipcc())), "amdclang++")
    return [compiler, f'-DSVDQ_TORCH_VERSION="{torch.__version__}"', "-O2", "-std=c++17", "-fPIC", "-shared", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
            *flags, os.path.join(CSRC, "host.cpp"), "-lc10", "-ltorch_cpu", "-ltorch_python", "-o", out]  # fmt: skip


def build(verbose: bool = False) -> str:
    def run(cmd: list[str]) -> None:
        if verbose:
            print(" ".join(cmd), flush=True)
        proc = subprocess.run(cmd, capture_output=True, text=True)
        err = "\n".join(ln for ln in proc.stderr.splitlines() if "not a recognized feature" not in ln)
        if proc.returncode != 0:
            raise RuntimeError(f"{cmd[0]} failed ({proc.returncode}):\n{err}")
        if verbose and err.strip():
            print(err, file=sys.stderr)

    # one compiler process per source file: the kernels' instantiations are what takes the time
    with tempfile.TemporaryDirectory() as tmp, ThreadPoolExecutor(min(len(SOURCES), os.cpu_count() or 1)) as pool:
        objs = [os.path.join(tmp, s + ".o") for s in SOURCES]
        list(pool.map(run, [[hipcc(), *FLAGS, "-c", os.path.join(CSRC, s), "-o", o] for s, o in zip(SOURCES, objs)] + [host_command(HOST + ".tmp")]))
        run([hipcc(), *FLAGS, "-shared", *objs, "-o", LIB + ".tmp"])
    os.replace(LIB + ".tmp", LIB)
    os.replace(HOST + ".tmp", HOST)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
