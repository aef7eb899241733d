"""Build recipe for libfastcache_hip.so (hipcc, gfx950 only) and _host.so (g++, against torch's headers).

``python -m fastcache_amd.build`` compiles every ``csrc/*.hip`` file into one shared library
next to this file, and ``csrc/fc_host.cpp`` (the host path that takes torch tensors) into a CPython module beside
it.  hipcc cross-compiles without a GPU, so both are built on the development host and travel with the source tree.
"""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
LIB_PATH = PKG_DIR / "libfastcache_hip.so"
HOST_SRC = CSRC / "fc_host.cpp"
HOST_PATH = PKG_DIR / "_host.so"
OBJ_DIR = PKG_DIR / "csrc" / "build"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
DEVICE_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-fPIC",
    "-std=c++17",
    # packed-fp32 instructions are kept out of every kernel of this library
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip"))


def _compile_one(src: Path, verbose: bool) -> Path:
    obj = OBJ_DIR / (src.stem + ".o")
    extra = os.environ.get("FC_EXTRA_HIPCC_FLAGS", "").split()      # e.g. -DCP_R=16 for tuning runs
    cmd = [HIPCC, *DEVICE_FLAGS, *extra, "-c", str(src), "-o", str(obj)]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{res.stdout}\n{res.stderr}")
    return obj


def _compile_host(verbose: bool) -> Path:
    import torch
    from torch.utils import cpp_extension
    obj = OBJ_DIR / "fc_host.o"
    includes = [*cpp_extension.include_paths(), "/opt/rocm/include", sysconfig.get_paths()["include"]]
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-fPIC", "-std=c++17", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *(f"-isystem{d}" for d in includes),
           "-c", str(HOST_SRC), "-o", str(obj)]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed on {HOST_SRC.name}:\n{res.stdout}\n{res.stderr}")
    return obj


def _link(cmd, target: Path, verbose: bool) -> None:
    tmp = target.with_suffix(".so.tmp")
    cmd = [*cmd, "-shared", "-fPIC", "-o", str(tmp)]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, target)


def _link_host(obj: Path, verbose: bool) -> None:
    """The module finds the kernel library beside itself; torch's libraries are loaded before it is imported."""
    from torch.utils import cpp_extension
    _link([os.environ.get("CXX", "g++"), str(obj), *(f"-L{d}" for d in cpp_extension.library_paths()), f"-L{PKG_DIR}",
           "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python", f"-l:{LIB_PATH.name}", "-Wl,-rpath,$ORIGIN"],
          HOST_PATH, verbose)


def build_library(verbose: bool = False, jobs: int = 4) -> Path:
    """Compile and link the library and the host module unconditionally; returns the library's path."""
    OBJ_DIR.mkdir(parents=True, exist_ok=True)
    srcs = sources()
    if not srcs:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        host = pool.submit(_compile_host, verbose)
        objs = list(pool.map(lambda s: _compile_one(s, verbose), srcs))
    _link([HIPCC, f"--offload-arch={ARCH}", *map(str, objs), "-Wl,-soname," + LIB_PATH.name], LIB_PATH, verbose)
    _link_host(host.result(), verbose)
    return LIB_PATH


if __name__ == "__main__":
    path = build_library(verbose="-q" not in sys.argv)
    print(f"built {path}")
