"""Build libcdx.so (the gfx950 HIP kernels behind include/cdx.h).

Every csrc/*.hip file is compiled on its own (in parallel) with hipcc for gfx950 and
the objects are linked into ``complexity_deep/libcdx.so``, next to the Python package
that loads it.  Objects go to ``<repo>/_build/``.  ``csrc/host/cdx_host.cpp``, the native
call paths of the operators, is compiled against torch's headers into
``complexity_deep/_host.so``, next to and linked to libcdx.so.

    python complexity-deep_amd/build_native.py
"""

from __future__ import annotations

import concurrent.futures as cf
import os
import subprocess
import sys
import sysconfig
from pathlib import Path

HERE = Path(__file__).resolve().parent
REPO = HERE.parent
CSRC = HERE / "csrc"
BUILD_DIR = REPO / "_build"
LIB_PATH = HERE / "complexity_deep" / "libcdx.so"
HOST_SRC = CSRC / "host" / "cdx_host.cpp"
HOST_PATH = HERE / "complexity_deep" / "_host.so"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
# Packed-FP32 VALU forms are disabled for all device code (see the build notes in
# the package documentation); the host pass prints a harmless "not recognized" note.
COMMON_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def _compile(src: Path) -> Path:
    obj = BUILD_DIR / (src.stem + ".o")
    cmd = [HIPCC, *COMMON_FLAGS, "-c", str(src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{res.stderr}")
    return obj


def _compile_host() -> Path:
    """Object of the host-only extension (it runs beside the kernels' compilation)."""
    import torch
    from torch.utils import cpp_extension

    obj = BUILD_DIR / "cdx_host.o"
    includes = [*cpp_extension.include_paths(), "/opt/rocm/include", sysconfig.get_paths()["include"]]
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *(f"-I{i}" for i in includes),
           "-c", str(HOST_SRC), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed for {HOST_SRC.name}:\n{res.stderr}")
    return obj


def _link_host(obj: Path) -> None:
    from torch.utils import cpp_extension

    tmp = HOST_PATH.with_suffix(".so.tmp")
    cmd = [os.environ.get("CXX", "g++"), "-shared", "-o", str(tmp), str(obj), f"-L{LIB_PATH.parent}", "-l:libcdx.so",
           *(f"-L{d}" for d in cpp_extension.library_paths()), "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python",
           "-Wl,-rpath,$ORIGIN"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    os.replace(tmp, HOST_PATH)


def build(verbose: bool = False) -> Path:
    """Compile every kernel source and link libcdx.so, and the host extension; returns the
    library path."""
    BUILD_DIR.mkdir(parents=True, exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    if not sources:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    workers = min(len(sources), max(1, min(16, os.cpu_count() or 1)))
    with cf.ThreadPoolExecutor(max_workers=workers) as ex:
        host = ex.submit(_compile_host)
        objs = list(ex.map(_compile, sources))
        host_obj = host.result()
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    os.replace(tmp, LIB_PATH)
    _link_host(host_obj)
    if verbose:
        print(f"built {LIB_PATH} from {len(objs)} sources, and {HOST_PATH.name}")
    return LIB_PATH


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
