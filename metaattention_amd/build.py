"""Builds the gfx950 kernel library and the host extension in-tree.

``python -m metaattention_amd.build`` (or ``build_library()``) compiles every
``csrc/*.hip`` translation unit for gfx950 and links
``metaattention_amd/lib/libmetaattention_hip.so``, then compiles
``csrc/host_ops.cpp`` (the operators' calls in native code) against this
PyTorch into ``metaattention_amd/lib/ma_host.so``.  hipcc cross-compiles, so no
GPU is needed to build.
"""
from __future__ import annotations

import concurrent.futures
import os
import subprocess
import sys
import warnings

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_DIR = os.path.join(HERE, "lib")
LIB_PATH = os.path.join(LIB_DIR, "libmetaattention_hip.so")
HOST_PATH = os.path.join(LIB_DIR, "ma_host.so")
OBJ_DIR = os.path.join(HERE, "build")

# -packed-fp32-ops: keep the compiler from forming v_pk_{add,mul,fma}_f32
HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffast-math", "-fno-finite-math-only",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]

# -amdgpu-mfma-vgpr-form: kernels of more than 256 registers otherwise put every MFMA's result in accumulation registers, the
# scores too, which the vector ALU then moves out one by one.  Forward + backward of B2 H32 S1600 256/256 causal by such kernels 711 us
# without, 614 with it
UNIT_FLAGS = {unit: ["-mllvm", "-amdgpu-mfma-vgpr-form"] for unit in ("attn_bwd_256.hip",)}


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.isabs(cand) and os.path.exists(cand) or not os.path.isabs(cand)):
            return cand
    raise RuntimeError("hipcc not found")


def _run(cmd: list, what: str, verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{what} failed:\n{res.stdout}\n{res.stderr}")


def _compile(src: str, verbose: bool) -> str:
    obj = os.path.join(OBJ_DIR, os.path.basename(src).replace(".hip", ".o"))
    cmd = [_hipcc(), *HIPCC_FLAGS, "-c", src, "-o", obj]
    extra = UNIT_FLAGS.get(os.path.basename(src), [])
    try:
        _run([*cmd, *extra], f"hipcc of {src}", verbose)
    except RuntimeError as e:
        # (an option of the compiler's own, which another version may not have: the kernels are right without it, and slower)
        if not extra or "nknown command line argument" not in str(e):
            raise
        warnings.warn(f"hipcc does not know {' '.join(extra)}: {os.path.basename(src)} is compiled without")
        _run(cmd, f"hipcc of {src}", verbose)
    return obj


def _compile_host(verbose: bool) -> str:
    import sysconfig
    import torch
    from torch.utils import cpp_extension
    obj = os.path.join(OBJ_DIR, "host_ops.o")
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-isystem", sysconfig.get_paths()["include"],
          *[x for d in cpp_extension.include_paths("cuda") for x in ("-isystem", d)],
          "-c", os.path.join(CSRC, "host_ops.cpp"), "-o", obj], "g++ of host_ops.cpp", verbose)
    return obj


def _link_host(obj: str, verbose: bool) -> None:
    from torch.utils import cpp_extension
    _run(["g++", "-shared", "-fPIC", "-o", HOST_PATH, obj, "-L", LIB_DIR, "-lmetaattention_hip", "-Wl,-rpath,$ORIGIN",
          *[f"-L{d}" for d in cpp_extension.library_paths("cuda")], "-ltorch_python", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip"],
         "link of ma_host.so", verbose)


def build_library(verbose: bool = False, jobs: int = 8) -> str:
    os.makedirs(LIB_DIR, exist_ok=True)
    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs = sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as ex:
        host_obj = ex.submit(_compile_host, verbose)
        objs = list(ex.map(lambda s: _compile(s, verbose), srcs))
        _run([_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB_PATH, *objs], "link", verbose)
        _link_host(host_obj.result(), verbose)
    return LIB_PATH


if __name__ == "__main__":
    print(build_library(verbose="-v" in sys.argv))
