"""Build libfusionmoe.so (the gfx950 kernels and their C ABI) in-tree with hipcc.

Usage: python -m fusionllm_amd.build   (or fusionllm_amd.build.build_library())

Every .hip file under csrc/ is compiled for gfx950 only and linked into one
shared library next to this file; csrc/block_host.cpp becomes the Python
module _block_host beside it.  Compiler flags of the kernels:
  -ffp-contract=off   every fused multiply-add in the kernels is explicit, so
                      the rounding steps are the written ones;
  -packed-fp32-ops off: some packed fp32 forms have given wrong results on
                      this hardware (hipcc's host pass warns that it does not
                      know the feature; harmless).
"""
from __future__ import annotations

import importlib.util
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
BUILD_DIR = PKG_DIR / "_build"
LIB_PATH = PKG_DIR / "libfusionmoe.so"
HOST_PATH = PKG_DIR / "_block_host.so"
ARCH = "gfx950"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
COMMON_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++20",
    "-fPIC",
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-command-line-argument",
]


# Per-source flags (none at present).
EXTRA_FLAGS: dict[str, list[str]] = {}


def _compile(src: Path) -> Path:
    obj = BUILD_DIR / (src.stem + ".o")
    cmd = [HIPCC, *COMMON_FLAGS, *EXTRA_FLAGS.get(src.name, []), "-c", str(src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{res.stdout}\n{res.stderr}")
    return obj


def build_host_module() -> Path:
    """Compile csrc/block_host.cpp (the block's launch sequence on torch's C++ API;
    it is given the entry points of the loaded library at run time) into the
    module _block_host."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    tmp = HOST_PATH.with_suffix(".so.tmp")
    includes = [*cpp_extension.include_paths(), sysconfig.get_path("include")]
    libdir = cpp_extension.library_paths()[0]
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall",
           "-DTORCH_EXTENSION_NAME=_block_host",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *[f"-I{i}" for i in includes], str(CSRC / "block_host.cpp"), "-o", str(tmp),
           f"-L{libdir}", "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed on block_host.cpp:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, HOST_PATH)
    return HOST_PATH


def build_library(verbose: bool = True) -> Path:
    """Compile every kernel source and link libfusionmoe.so; where torch is installed, build
    the host module too (the library and its C ABI need neither torch nor a host compiler).
    Returns the library's path."""
    BUILD_DIR.mkdir(exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    if not sources:
        raise RuntimeError(f"no kernel sources under {CSRC}")
    with ThreadPoolExecutor(max_workers=min(8, len(sources))) as pool:
        objs = list(pool.map(_compile, sources))
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, LIB_PATH)
    if importlib.util.find_spec("torch") is not None:
        build_host_module()
    if verbose:
        print(f"built {LIB_PATH} from {len(sources)} sources", file=sys.stderr)
    return LIB_PATH


if __name__ == "__main__":
    build_library()
