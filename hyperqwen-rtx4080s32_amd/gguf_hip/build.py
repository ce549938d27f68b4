"""Builds the HIP library ``libgqk.so`` in-tree for gfx950 (hipcc, no JIT cache).

    python hyperqwen-rtx4080s32_amd/gguf_hip/build.py     # as a script: no package import, so a
                                                          # stale or missing library is no obstacle
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)                      # hyperqwen-rtx4080s32_amd/
REPO = os.path.dirname(ROOT)
CSRC = os.path.join(ROOT, "csrc")
BUILD = os.path.join(ROOT, "_build")
LIB = os.path.join(PKG, "libgqk.so")
# (source, extra flags, object): the GEMM is compiled once per token-block count, side by side
SOURCES = (("gqk_api.hip", (), "gqk_api.o"), ("gqk_codec.hip", (), "gqk_codec.o"), ("gqk_gemv.hip", (), "gqk_gemv.o"),
           ("gqk_mid.hip", (), "gqk_mid.o"), ("gqk_gemm_plan.hip", (), "gqk_gemm_plan.o"),
           *(("gqk_gemm.hip", (f"-DGQK_GEMM_MB={mb}",), f"gqk_gemm{mb}.o") for mb in (2, 4, 8)),
           ("gqk_gguf.cpp", (), "gqk_gguf.o"))
ARCH = os.environ.get("GQK_OFFLOAD_ARCH", "gfx950")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "-O3", "-fPIC", "-std=c++17", f"--offload-arch={ARCH}",
    "-I", os.path.join(REPO, "include"), "-I", CSRC,
    # packed fp32 VALU ops stay off (the pool's boxes have shown silent errors from them)
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # MFMA accumulators in ordinary VGPRs (no v_accvgpr_read round trips in the GEMV epilogue)
    "-mllvm", "-amdgpu-mfma-vgpr-form",
]


def _run(cmd: list[str]) -> None:
    p = subprocess.run(cmd, capture_output=True, text=True)
    if p.returncode != 0:
        raise RuntimeError(f"hipcc failed ({p.returncode}): {' '.join(cmd)}\n{p.stderr[-6000:]}")


def build(jobs: int | None = None) -> str:
    """Compile every source (HIP kernels; the host-only GGUF reader) and link libgqk.so (always rebuilds); returns the library path."""
    os.makedirs(BUILD, exist_ok=True)
    objs = []
    cmds = []
    for src, extra, name in SOURCES:
        obj = os.path.join(BUILD, name)
        objs.append(obj)
        cmds.append([HIPCC, *FLAGS, *extra, "-c", os.path.join(CSRC, src), "-o", obj])
    with ThreadPoolExecutor(max_workers=jobs or min(len(cmds), os.cpu_count() or 4)) as ex:
        list(ex.map(_run, cmds))
    tmp = LIB + ".tmp"
    _run([HIPCC, "-shared", f"--offload-arch={ARCH}", "-o", tmp, *objs])
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(int(sys.argv[1]) if len(sys.argv) > 1 else None))
