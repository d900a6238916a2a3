"""Build recipe: compiles the HIP sources into ``libcueq_amd.so`` for gfx950 with hipcc.

The host module (``csrc/host/*.cpp``, launch paths and autograd functions against PyTorch's C++ interface) is built next
to it as ``_host.so``.  ``python -m cuequivariance_amd.build`` (or ``__graft_entry__.build()``) compiles every
translation unit to an object file in ``cuequivariance_amd/_build`` (in parallel, only
the stale ones unless ``force``) and links them.  Cross-compiles without a GPU.
"""

from __future__ import annotations

import concurrent.futures
import os
import shutil
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
BUILD = PKG / "_build"
LIB = PKG / "libcueq_amd.so"

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

# Packed fp32 instructions are disabled for every device compile of this library.
COMMON_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    "-Werror=return-type",  # (device code that runs off the end of a function goes on into whatever follows it)
    f"-I{ROOT / 'include'}",
    f"-I{CSRC}",
]


def sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip")) + sorted((CSRC / "generated").glob("*.hip"))


def _stale(src: Path, obj: Path) -> bool:
    if not obj.exists():
        return True
    newest = max([src.stat().st_mtime] + [h.stat().st_mtime for h in list(CSRC.glob("*.h")) + [ROOT / "include" / "cueq_amd.h"]])
    return obj.stat().st_mtime < newest


def _compile(src: Path, obj: Path) -> None:
    cmd = [HIPCC, *COMMON_FLAGS, "-c", str(src), "-o", str(obj)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{r.stdout}\n{r.stderr}")


HOST = PKG / "_host.so"


def build_host(force: bool = False) -> Path:
    """The host module (``csrc/host``): C++ against PyTorch's headers, no device code; it loads the library at run time."""
    import sysconfig

    import torch

    src_dir = CSRC / "host"
    srcs = sorted(src_dir.glob("*.cpp"))
    headers = [*src_dir.glob("*.h"), ROOT / "include" / "cueq_amd.h"]
    torch_dir = Path(torch.__file__).resolve().parent
    flags = ["-std=c++17", "-O2", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM", "-DTORCH_EXTENSION_NAME=_host", "-DTORCH_API_INCLUDE_EXTENSION_H",
             f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f"-I{ROOT / 'include'}", f"-I{torch_dir / 'include'}",
             f"-I{torch_dir / 'include' / 'torch' / 'csrc' / 'api' / 'include'}", "-isystem", "/opt/rocm/include", f"-I{sysconfig.get_paths()['include']}"]
    todo = []
    for s in srcs:
        obj = BUILD / f"host_{s.stem}.o"
        if force or not obj.exists() or obj.stat().st_mtime < max(f.stat().st_mtime for f in [s, *headers]):
            todo.append((s, obj))

    def compile_one(s, obj):
        r = subprocess.run(["g++", *flags, "-c", str(s), "-o", str(obj)], capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"g++ failed for {s.name}:\n{r.stderr[-4000:]}")

    with concurrent.futures.ThreadPoolExecutor(max_workers=4) as ex:
        for f in [ex.submit(compile_one, s, o) for s, o in todo]:
            f.result()
    if todo or not HOST.exists():
        libs = torch_dir / "lib"
        r = subprocess.run(["g++", "-shared", "-o", str(HOST), *[str(BUILD / f"host_{s.stem}.o") for s in srcs], f"-L{libs}", f"-Wl,-rpath,{libs}",
                            "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip", "-ltorch_python", "-ldl"], capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"link of the host module failed:\n{r.stderr[-4000:]}")
    return HOST


def build_library(force: bool = False, jobs: int | None = None, verbose: bool = True) -> Path:
    BUILD.mkdir(exist_ok=True)
    sys.path.insert(0, str(ROOT))
    from cuequivariance_amd.codegen import registry as _registry

    _registry.generate()
    srcs = sources()
    todo = []
    for s in srcs:
        obj = BUILD / (s.stem + ".o")
        if force or _stale(s, obj):
            todo.append((s, obj))
    jobs = jobs or min(8, max(1, (os.cpu_count() or 2)))
    if verbose and todo:
        print(f"[cueq_amd] compiling {len(todo)} file(s) for gfx950", file=sys.stderr, flush=True)
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as ex:
        for f in [ex.submit(_compile, s, o) for s, o in todo]:
            f.result()
    objs = [str(BUILD / (s.stem + ".o")) for s in srcs]
    if todo or not LIB.exists():
        cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(LIB), *objs]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    build_host(force)
    # fused kernels of the registered fully connected products: separate small objects next to the library
    from cuequivariance_amd import jit as _jit

    _jit.prebuild_fully_connected(force)
    return LIB


if __name__ == "__main__":
    build_library(force="--force" in sys.argv)
    print(LIB)
