"""Build liblatentq_hip.so (gfx950) and the Python binding _lqbind.so in-tree.

`python -m latentq_llm_amd.build` compiles every HIP translation unit under
``csrc/`` with hipcc, links the C-ABI shared library next to this file, and
compiles ``csrc/lq_bind.cpp`` (host code) against it and torch's headers. hipcc
cross-compiles without a GPU, so this runs anywhere ROCm is installed.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(CSRC, "obj")
LIB = os.path.join(HERE, "liblatentq_hip.so")
BIND = os.path.join(HERE, "_lqbind.so")

ARCH = "gfx950"
# Packed-FP32 VALU instructions are disabled for every device translation unit.
COMMON = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # every fp32 rounding is written out (fmaf where a fused operation is meant)
    "-ffp-contract=off",
    # up to 16 (14 in practice) dwords of leading scalar arguments arrive in registers with the wave instead of by a load that
    # every address waits for: 0.1 to 0.4 us of a 3 to 12 us kernel. Arguments passed as a structure are not preloaded.
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
    "-Wno-unused-command-line-argument", "-Wno-unknown-warning-option",
]
EXTRA: dict[str, list[str]] = {}


def hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found (need ROCm to build liblatentq_hip.so)")
    return exe


def sources() -> list[str]:
    return sorted(f for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(src: str) -> str:
    obj = os.path.join(OBJ, src[:-4] + ".o")
    cmd = [hipcc(), *COMMON, *EXTRA.get(src, []), "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{r.stdout}\n{r.stderr}")
    return obj


def _compile_binding(out: str) -> str:
    """lq_bind.cpp to an object: plain host C++ that sees HIP's and torch's headers."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *(f"-I{d}" for d in include_paths("cuda")), f"-I{sysconfig.get_paths()['include']}",
           "-c", os.path.join(CSRC, "lq_bind.cpp"), "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed on lq_bind.cpp:\n{r.stdout}\n{r.stderr}")
    return out


def _link_binding(obj: str) -> None:
    import torch
    libs = os.path.join(os.path.dirname(torch.__file__), "lib")
    tmp = BIND + ".tmp"
    cmd = ["g++", "-shared", "-o", tmp, obj, f"-L{HERE}", f"-l:{os.path.basename(LIB)}", f"-L{libs}", "-ltorch_python", "-ltorch",
           "-lc10", "-ltorch_hip", "-lc10_hip", "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"linking _lqbind.so failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, BIND)


def build_library(verbose: bool = True, jobs: int = 8) -> str:
    os.makedirs(OBJ, exist_ok=True)
    srcs = sources()
    with ThreadPoolExecutor(max_workers=min(jobs, len(srcs) + 1)) as ex:
        bind = ex.submit(_compile_binding, os.path.join(OBJ, "lq_bind.o"))
        objs = list(ex.map(_compile, srcs))
    tmp = LIB + ".tmp"
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-fno-gpu-rdc", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    _link_binding(bind.result())
    if verbose:
        print(f"built {LIB} from {len(srcs)} sources, and {BIND}", file=sys.stderr)
    return LIB


if __name__ == "__main__":
    build_library()
