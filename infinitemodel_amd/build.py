"""Build libimq.so (the gfx950 HIP kernels + C ABI) in-tree with hipcc.

Usage: ``python -m infinitemodel_amd.build`` (or ``__graft_entry__.build()``). Each ``csrc/*.hip``
is compiled to an object in parallel, then linked into ``infinitemodel_amd/_lib/libimq.so``; the native
host path of the eager calls (``csrc/fastcall.cpp``) becomes ``infinitemodel_amd/_lib/imq_fast.so``.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT_DIR = os.path.join(HERE, "_lib")
OBJ_DIR = os.path.join(HERE, "_lib", "obj")
LIB = os.path.join(OUT_DIR, "libimq.so")
FAST = os.path.join(OUT_DIR, "imq_fast.so")
ARCH = os.environ.get("IMQ_OFFLOAD_ARCH", "gfx950")

# Packed-fp32 VALU ops are disabled for all device code (hipcc flag; the host pass ignores it).
COMMON = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def hipcc() -> str:
    for c in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if c and os.path.exists(c):
            return c
    raise RuntimeError("hipcc not found (ROCm toolchain required to build libimq.so)")


# Per-source extra flags. moe_rb.hip: MFMA results in VGPRs (LLVM's VGPR form of the MFMA
# instructions), so the folded MoE kernels' per-group fold reads them without AGPR copies and two
# waves fit per SIMD; the option is scoped to that file's kernels.
EXTRA = {"moe_rb.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"]}


def _compile(src: str) -> str:
    obj = os.path.join(OBJ_DIR, os.path.basename(src).replace(".hip", ".o"))
    cmd = [hipcc(), *COMMON, *EXTRA.get(os.path.basename(src), []), "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr}")
    return obj


def _build_fast() -> None:
    """The native host path of the eager calls (csrc/fastcall.cpp): a CPython module against torch's
    headers and the interpreter's, no device code."""
    import sysconfig

    import torch
    root = os.path.dirname(torch.__file__)
    inc = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
           os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"), sysconfig.get_paths()["include"]]
    tmp = FAST + ".tmp"
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-DUSE_ROCM", "-D__HIP_PLATFORM_AMD__=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *(f"-I{d}" for d in inc),
           os.path.join(CSRC, "fastcall.cpp"), "-o", tmp, "-L" + os.path.join(root, "lib"), "-lc10", "-lc10_hip",
           "-ltorch_cpu", "-ltorch_python"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed for fastcall.cpp:\n{r.stderr}")
    os.replace(tmp, FAST)


def build(verbose: bool = True) -> str:
    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs = sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))
    with cf.ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        fast = ex.submit(_build_fast)
        objs = list(ex.map(_compile, srcs))
        fast.result()
    tmp = LIB + ".tmp"
    cmd = [hipcc(), *COMMON, "-shared", *objs, "-o", tmp]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"[imq] built {LIB} ({len(srcs)} sources, {ARCH})", flush=True)
    return LIB


if __name__ == "__main__":
    build()
    sys.exit(0)
