"""Compile the gfx950 C-ABI library ``lib/libmegalodon_hip.so`` with hipcc and the
host extension ``_host`` with g++.

The library has no PyTorch dependency: it is plain HIP behind ``extern "C"``
entry points (``include/megalodon_hip.h``), so a single ``hipcc -shared``
invocation per translation unit is its whole build.  The host extension is the
C++ part of the Python package (``csrc/host``): it links the library and the
installed PyTorch and holds no kernels.
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
LIB_DIR = PKG_DIR / "lib"
LIB_PATH = LIB_DIR / "libmegalodon_hip.so"

HOST_SRC = CSRC / "host"
HOST_PATH = PKG_DIR / ("_host" + sysconfig.get_config_var("EXT_SUFFIX"))

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
# packed-fp32 VALU forms are disabled for every device translation unit
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument", "-Wno-unknown-warning-option",
    "-Wno-ignored-optimization-argument",
]


def sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip"))


def _compile(src: Path, obj_dir: Path, extra: list[str], force: bool = True) -> Path:
    obj = obj_dir / (src.stem + ".o")
    if not force and obj.exists():
        deps = [src, *CSRC.glob("*.hpp"), PKG_DIR.parent / "include" / "megalodon_hip.h"]
        if all(obj.stat().st_mtime > d.stat().st_mtime for d in deps):
            return obj
    cmd = [HIPCC, *FLAGS, *extra, "-c", str(src), "-o", str(obj)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{r.stdout}\n{r.stderr}")
    return obj


def build_library(verbose: bool = True, extra: list[str] | None = None, jobs: int = 8,
                  force: bool = True) -> Path:
    """Compile every ``csrc/*.hip`` and link ``libmegalodon_hip.so``.  With
    ``force=False`` objects newer than their source and the shared headers are
    reused (developer iterations only)."""
    extra = list(extra or [])
    obj_dir = PKG_DIR / "build"
    obj_dir.mkdir(exist_ok=True)
    LIB_DIR.mkdir(exist_ok=True)
    srcs = sources()
    if verbose:
        print(f"[megalodon_amd] hipcc {ARCH}: {', '.join(s.name for s in srcs)}", flush=True)
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(lambda s: _compile(s, obj_dir, extra, force), srcs))
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB_PATH)
    if verbose:
        print(f"[megalodon_amd] built {LIB_PATH}", flush=True)
    return LIB_PATH


def _torch_dir() -> Path:
    import importlib.util
    return Path(importlib.util.find_spec("torch").origin).parent


def build_host(verbose: bool = True, jobs: int = 8, force: bool = True) -> Path:
    """Compile ``csrc/host/*.cpp`` and link the extension module ``megalodon_amd._host``
    (after ``build_library``, whose shared library it links)."""
    torch_dir = _torch_dir()
    obj_dir = PKG_DIR / "build"
    obj_dir.mkdir(exist_ok=True)
    srcs = sorted(HOST_SRC.glob("*.cpp"))
    rocm = Path(HIPCC).parent.parent
    flags = ["-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
             "-DTORCH_EXTENSION_NAME=_host", f"-I{torch_dir}/include", f"-I{torch_dir}/include/torch/csrc/api/include",
             f"-I{rocm}/include", f"-I{sysconfig.get_paths()['include']}"]
    if verbose:
        print(f"[megalodon_amd] g++: {', '.join(s.name for s in srcs)}", flush=True)

    def compile_one(src: Path) -> Path:
        obj = obj_dir / ("host_" + src.stem + ".o")
        deps = [src, *HOST_SRC.glob("*.hpp"), PKG_DIR.parent / "include" / "megalodon_hip.h"]
        if force or not obj.exists() or any(obj.stat().st_mtime <= d.stat().st_mtime for d in deps):
            r = subprocess.run(["g++", *flags, "-c", str(src), "-o", str(obj)], capture_output=True, text=True)
            if r.returncode != 0:
                raise RuntimeError(f"g++ failed on {src.name}:\n{r.stdout}\n{r.stderr}")
        return obj

    with ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(compile_one, srcs))
    tmp = HOST_PATH.with_suffix(".so.tmp")
    cmd = ["g++", "-shared", "-o", str(tmp), *map(str, objs), f"-L{LIB_DIR}", "-lmegalodon_hip",
           "-Wl,-rpath,$ORIGIN/lib", f"-L{torch_dir}/lib", "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, HOST_PATH)
    if verbose:
        print(f"[megalodon_amd] built {HOST_PATH}", flush=True)
    return HOST_PATH


if __name__ == "__main__":
    args = sys.argv[1:]
    incremental = "--incremental" in args
    build_library(extra=[a for a in args if a != "--incremental"], force=not incremental)
    build_host(force=not incremental)
