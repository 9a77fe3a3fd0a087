"""Builds libtileinfer_amd.so (the gfx950 kernels + C ABI) in-tree with hipcc, and _pycalls.so (the
Python entry points' common form in native code, csrc/pycalls.cpp) with the host compiler.

Usage: ``python -m tileinfer_amd.build`` (or ``tileinfer_amd.build.build()``). Both land next to this
file, where :mod:`tileinfer_amd._lib` loads them; object files go to ``_build/``. Cross-compiles on a
host without a GPU.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import sysconfig
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
BUILD_DIR = PKG_DIR / "_build"
LIB_NAME = "libtileinfer_amd.so"
LIB_PATH = PKG_DIR / LIB_NAME
CALLS_PATH = PKG_DIR / "_pycalls.so"

ARCH = os.environ.get("TI_OFFLOAD_ARCH", "gfx950")

# -packed-fp32-ops: keep the compiler from forming v_pk_{add,mul,fma}_f32.
HIP_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Wno-unused-command-line-argument",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-mcode-object-version=5",
]


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (set HIPCC or install ROCm)")


def sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip"))


def _compile(hipcc: str, src: Path, extra: list[str]) -> Path:
    obj = BUILD_DIR / (src.stem + ".o")
    cmd = [hipcc, *HIP_FLAGS, *extra, "-c", str(src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    # The host pass does not know the packed-fp32 feature and says so; drop only that line.
    noise = "'-packed-fp32-ops' is not a recognized feature"
    err = "\n".join(l for l in res.stderr.splitlines() if noise not in l)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{' '.join(cmd)}\n{err}")
    if err.strip():
        print(err, file=sys.stderr)
    return obj


def _cxx() -> str | None:
    """A host C++ compiler; ROCm's own where there is no other."""
    rocm = Path(_hipcc()).resolve().parent.parent
    for cand in (os.environ.get("CXX"), shutil.which("g++"), shutil.which("clang++"),
                 str(rocm / "bin" / "amdclang++"), str(rocm / "llvm" / "bin" / "clang++")):
        if cand and (os.path.exists(cand) or shutil.which(cand)):
            return cand
    return None


def _build_calls() -> None:
    """csrc/pycalls.cpp against torch's and Python's headers (host code only). Where a host compiler or
    the headers are missing it is left out, with a line that says so: the entry points then run their
    Python form."""
    import torch
    from torch.utils import cpp_extension

    from ._lib import versions

    cxx = _cxx()
    includes = [*cpp_extension.include_paths(), sysconfig.get_paths()["include"]]
    missing = [n for n in ("ATen/ATen.h", "Python.h")
               if not any(os.path.exists(os.path.join(p, n)) for p in includes)]
    missing += [] if cxx else ["a host C++ compiler"]
    if missing:
        CALLS_PATH.unlink(missing_ok=True)
        print(f"{CALLS_PATH.name} left out ({', '.join(missing)} not found): calls take 5 to 10 us more "
              "of host time", file=sys.stderr)
        return
    tmp = CALLS_PATH.with_suffix(".so.tmp")
    lib_dir = Path(torch.__file__).resolve().parent / "lib"
    cmd = [cxx, "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall",
           f'-DTI_BUILT_FOR="{versions()}"', f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *(f"-isystem{p}" for p in includes), str(CSRC / "pycalls.cpp"), "-o", str(tmp),
           f"-L{lib_dir}", "-ltorch_python", "-ltorch_cpu", "-lc10"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"host compiler failed on pycalls.cpp:\n{' '.join(cmd)}\n{res.stderr}")
    if res.stderr.strip():
        print(res.stderr, file=sys.stderr)
    os.replace(tmp, CALLS_PATH)


def build(verbose: bool = True, extra_flags: list[str] | None = None) -> Path:
    """Compile every csrc/*.hip for gfx950 and link libtileinfer_amd.so, and compile _pycalls.so.
    Always rebuilds."""
    hipcc = _hipcc()
    BUILD_DIR.mkdir(exist_ok=True)
    extra = list(extra_flags or [])
    srcs = sources()
    with cf.ThreadPoolExecutor(max_workers=min(8, len(srcs) + 1)) as ex:
        calls = ex.submit(_build_calls)
        objs = list(ex.map(lambda s: _compile(hipcc, s, extra), srcs))
        calls.result()
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{' '.join(cmd)}\n{res.stderr}")
    os.replace(tmp, LIB_PATH)
    if verbose:
        print(f"built {LIB_PATH} from {len(srcs)} sources for {ARCH}")
    return LIB_PATH


if __name__ == "__main__":
    build()
