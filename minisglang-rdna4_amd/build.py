"""Build libw4a8_mi355x.so (gfx950) from csrc/*.hip and w4a8_host.so (the operators' host path, no device
code) from csrc/host.cpp, both with hipcc, in-tree.

Objects compile in parallel into _build/, the shared library lands in _lib/. Every call
recompiles (the build is the "does it build" check), so keep it cheap: one object per source.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
BUILD = PKG / "_build"
LIBDIR = PKG / "_lib"
LIBNAME = "libw4a8_mi355x.so"
ARCH = os.environ.get("W4A8_OFFLOAD_ARCH", "gfx950")

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # no packed-FP32 VALU forms anywhere in device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
]


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.sep not in cand or os.path.exists(cand)):
            return cand
    raise RuntimeError("hipcc not found")


def _compile(src: Path) -> Path:
    obj = BUILD / (src.stem + ".o")
    cmd = [_hipcc(), *HIPCC_FLAGS, "-c", str(src), "-o", str(obj)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{r.stderr[-4000:]}")
    return obj


def _build_host() -> Path:
    """csrc/host.cpp against the installed torch's C++ libraries (loaded before it at run time). It records
    the torch and Python it was built for; _host.py uses it with those only."""
    import sysconfig

    import torch

    tdir = Path(torch.__file__).resolve().parent
    out = LIBDIR / "w4a8_host.so"
    tmp = out.with_suffix(".so.tmp")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    built_for = f"torch {torch.__version__}, Python {sys.version_info.major}.{sys.version_info.minor}"
    cmd = [_hipcc(), "-no-hip-rt", "-x", "c++", "-O2", "-std=c++17", "-shared", "-fPIC", "-fvisibility=hidden",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f'-DW4A8_BUILT_FOR="{built_for}"',
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
           f"-I{tdir / 'include'}", f"-I{tdir / 'include' / 'torch' / 'csrc' / 'api' / 'include'}", f"-I{rocm}/include",
           f"-I{sysconfig.get_paths()['include']}", str(CSRC / "host.cpp"), "-o", str(tmp), f"-L{tdir / 'lib'}",
           "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed for host.cpp:\n{r.stderr[-4000:]}")
    os.replace(tmp, out)
    return out


def lib_path() -> Path:
    return LIBDIR / LIBNAME


def build(verbose: bool = False) -> Path:
    BUILD.mkdir(exist_ok=True)
    LIBDIR.mkdir(exist_ok=True)
    srcs = sorted(CSRC.glob("*.hip"))
    jobs = min(len(srcs), max(1, min(8, os.cpu_count() or 1)))
    with cf.ThreadPoolExecutor(jobs) as ex:
        host = ex.submit(_build_host)
        objs = list(ex.map(_compile, srcs))
    out = lib_path()
    tmp = out.with_suffix(".so.tmp")
    cmd = [_hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr[-4000:]}")
    os.replace(tmp, out)
    host.result()  # after the link: the kernel library serves without the extension too
    if verbose:
        print(f"built {out}")
    return out


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
