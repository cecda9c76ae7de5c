"""Build recipe of the HIP library ``nanoquant_amd/libnq_hip.so`` (gfx950) and of
``nanoquant_amd/libnq_ops.so``, the C++ implementations of the torch operators.

``python -m nanoquant_amd.build`` compiles every source under ``csrc/`` with hipcc
and ``csrc/torch_ops/`` with g++ against torch's headers, and links the shared
libraries in place, next to this file, so that they travel with the source tree.
Objects go to ``_build/`` (git-ignored).
"""
from __future__ import annotations

import concurrent.futures
import hashlib
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD_DIR = os.path.join(os.path.dirname(HERE), "_build")
LIB_NAME = "libnq_hip.so"
LIB_PATH = os.path.join(HERE, LIB_NAME)
HEADER = os.path.join(os.path.dirname(HERE), "include", "nq_hip.h")
OPS_SOURCE = os.path.join(CSRC, "torch_ops", "nq_ops.cpp")
OPS_PATH = os.path.join(HERE, "libnq_ops.so")
ARCH = os.environ.get("NQ_OFFLOAD_ARCH", "gfx950")

COMMON_FLAGS = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
    # never let the compiler form packed fp32 VALU ops
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
    # a waves-per-EU hint the register allocator cannot meet is a tuning choice, not a defect
    "-Wno-pass-failed",
]


# Per-source additions. The GEMV source keeps MFMA accumulators in VGPRs (the VGPR form of the
# instruction): with the AGPR form the register allocator moved the batched kernels'
# accumulators between AGPRs and VGPRs on every loop trip (more such moves than MFMAs).
FILE_FLAGS = {
    "nq_gemv.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
}


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(path):
        raise RuntimeError("hipcc not found: the HIP library cannot be built")
    return path


def header_digest() -> str:
    """Define of the C ABI's digest, by which the two libraries tell that they were built from the same header."""
    with open(HEADER, "rb") as f:
        return f'-DNQ_HEADER_DIGEST="{hashlib.sha256(f.read()).hexdigest()[:16]}"'


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith((".hip", ".cpp")))


def _compile(src: str) -> str:
    obj = os.path.join(BUILD_DIR, os.path.basename(src) + ".o")
    cmd = [hipcc(), *COMMON_FLAGS, *FILE_FLAGS.get(os.path.basename(src), []), header_digest(), "-x", "hip", "-c", src,
           "-o", obj]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{proc.stdout}\n{proc.stderr}")
    # the host pass does not know the packed-fp32 feature and says so; nothing else is expected
    noise = [ln for ln in proc.stderr.splitlines() if "packed-fp32-ops" not in ln and ln.strip()]
    if noise:
        print("\n".join(noise), file=sys.stderr)
    return obj


def build_ops() -> str:
    """Compile the torch operators (host code only); returns the library's path."""
    import torch
    from torch.utils import cpp_extension

    lib_dir = os.path.join(os.path.dirname(torch.__file__), "lib")
    tmp = OPS_PATH + ".tmp"
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", header_digest()]
    for path in cpp_extension.include_paths("cuda"):
        cmd += ["-isystem", path]
    cmd += [OPS_SOURCE, "-o", tmp, f"-L{lib_dir}", "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{proc.stdout}\n{proc.stderr}")
    os.replace(tmp, OPS_PATH)
    return OPS_PATH


def build(verbose: bool = True) -> str:
    """Compile and link the libraries; returns the HIP library's path."""
    os.makedirs(BUILD_DIR, exist_ok=True)
    srcs = sources()
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, len(srcs) + 1)) as ex:
        ops = ex.submit(build_ops)
        objs = list(ex.map(_compile, srcs))
        ops.result()
    tmp = LIB_PATH + ".tmp"
    cmd = [hipcc(), "-shared", "-fPIC", f"--offload-arch={ARCH}", *objs, "-o", tmp]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed: {' '.join(cmd)}\n{proc.stdout}\n{proc.stderr}")
    os.replace(tmp, LIB_PATH)
    if verbose:
        print(f"built {LIB_PATH} from {len(srcs)} sources for {ARCH}")
    return LIB_PATH


if __name__ == "__main__":
    build()
