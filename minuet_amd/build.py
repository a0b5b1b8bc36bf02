"""Builds libminuet_hip.so (the C-ABI library of hand-written gfx950 kernels)
in-tree with hipcc.  ``python -m minuet_amd.build`` rebuilds it."""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

_HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(_HERE, "csrc")
LIB_DIR = os.path.join(_HERE, "lib")
LIB_PATH = os.path.join(LIB_DIR, "libminuet_hip.so")
HOST_PATH = os.path.join(LIB_DIR, "minuet_host.so")
SOURCES = ["runtime.hip", "sort.hip", "unique.hip", "points.hip", "query.hip", "pass.hip", "conv.hip", "implicit.hip", "compact.hip", "tiles.hip", "tiled_half.hip", "tiled_bf16.hip", "streamed_half.hip", "streamed_bf16.hip", "single.hip", "lookahead.hip"]
ARCH = "gfx950"
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    # packed fp32 instructions are kept out of every kernel on purpose
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.isabs(cand) and os.path.exists(cand) or not os.path.isabs(cand)):
            return cand
    return "hipcc"


def _compile(src: str) -> str:
    obj = os.path.join(LIB_DIR, os.path.splitext(src)[0] + ".o")
    cmd = [_hipcc(), *FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{proc.stdout}\n{proc.stderr}")
    return obj


def build_host() -> str:
    """Compile the Python extension module with the host side of layer calls
    (csrc/host.cpp, plain C++ against torch's headers)."""
    import sysconfig
    import torch
    from torch.utils.cpp_extension import include_paths
    os.makedirs(LIB_DIR, exist_ok=True)
    libraries = os.path.join(os.path.dirname(torch.__file__), "lib")
    # NDEBUG leaves out pybind11's thread-local reference counter.  A module with
    # thread-local data that nothing reads makes glibc (before 2.39) take the slow
    # way to everybody else's from the moment it is loaded: every torch operation
    # of the process took 20 % longer on the host.
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-DNDEBUG", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
           "-DUSE_ROCM", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *[f"-I{path}" for path in include_paths()], f"-I{sysconfig.get_paths()['include']}",
           f"-I{os.path.join(os.environ.get('ROCM_PATH', '/opt/rocm'), 'include')}",
           os.path.join(CSRC, "host.cpp"), "-o", HOST_PATH, f"-L{libraries}", "-ltorch_python", "-ltorch_cpu",
           "-ltorch_hip", "-lc10", "-lc10_hip"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed on host.cpp:\n{proc.stdout}\n{proc.stderr}")
    return HOST_PATH


def build_library(verbose: bool = True, host: bool = True) -> str:
    """Compile every HIP source, link the shared library and build the host
    extension (``host``).  Always rebuilds; the library is there also where the
    extension cannot be built, which is reported last."""
    os.makedirs(LIB_DIR, exist_ok=True)
    with ThreadPoolExecutor(max_workers=min(8, len(SOURCES) + 1)) as pool:
        extension = pool.submit(build_host) if host else None
        objects = list(pool.map(_compile, SOURCES))
    cmd = [_hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *objects, "-o", LIB_PATH]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed:\n{proc.stdout}\n{proc.stderr}")
    if verbose:
        print(f"built {LIB_PATH}", file=sys.stderr)
    if extension is not None:
        extension.result()
    return LIB_PATH


if __name__ == "__main__":
    build_library()
