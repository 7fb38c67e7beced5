"""Build libint4_hip.so (gfx950) in-tree with hipcc, and _int4_torch.so (host) with g++.

    python itmo-final-project_amd/build_lib.py [--jobs N]

Every call recompiles every source (object files go to ``_build/``, the
library to ``int4_hip/libint4_hip.so``, the torch binding of the Python entry
points' fast path to ``int4_hip/_int4_torch.so``).  hipcc cross-compiles for gfx950 on a
machine without a GPU.
"""
from __future__ import annotations

import argparse
import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

HERE = Path(__file__).resolve().parent
ROOT = HERE.parent
CSRC = HERE / "csrc"
BUILD = HERE / "_build"
LIB = HERE / "int4_hip" / "libint4_hip.so"
# measurement helpers for bench.py (not part of the library)
BENCH_SRC = CSRC / "bench"
BENCH_LIB = HERE / "int4_hip" / "libw4_bench.so"
# the Python entry points' native call path (built against the installed torch)
EXT_SRC = CSRC / "torch_ext" / "int4_torch.cpp"
EXT_LIB = HERE / "int4_hip" / "_int4_torch.so"
ARCH = "gfx950"

COMMON_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # Packed fp32 VALU instructions stay off: ordinary float code only.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", str(ROOT / "include"),
    "-I", str(CSRC),
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found (ROCm not installed?)")


def sources() -> list[Path]:
    return sorted(list(CSRC.glob("*.hip")) + list(CSRC.glob("*.cpp")))


def _compile(src: Path) -> Path:
    obj = BUILD / ((src.parent.name + "_" if src.parent == BENCH_SRC else "") + src.stem + ".o")
    cmd = [hipcc(), *COMMON_FLAGS, "-c", str(src), "-o", str(obj)]
    if src.suffix == ".cpp":
        cmd = [hipcc(), "-O3", "-std=c++17", "-fPIC", "-I", str(ROOT / "include"), "-I", str(CSRC),
               "-c", str(src), "-o", str(obj)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed: {src.name}\n{' '.join(cmd)}\n{err}")
    return obj


def build_ext() -> Path | None:
    """Compile int4_hip/_int4_torch.so (host code only) against the installed torch;
    None, and no binding, without torch or g++ (the library itself needs neither)."""
    import sysconfig

    try:
        import torch
    except ImportError:
        torch = None
    gxx = shutil.which("g++")
    if torch is None or gxx is None:
        print(f"{EXT_LIB.name} not built: {'g++' if torch else 'torch'} not found", file=sys.stderr)
        EXT_LIB.unlink(missing_ok=True)
        return None
    root = Path(torch.__file__).resolve().parent
    tmp = EXT_LIB.with_suffix(".so.tmp")
    # NDEBUG: without it pybind11's headers bring a thread-local counter.  A library
    # loaded with thread-local storage that a thread never touches leaves that
    # thread's table behind the loader's, and glibc (2.35 here) then takes
    # the slow path of every other thread-local access: torch.empty on the GPU took
    # 1.69 us instead of 1.37, every torch call of the process in proportion.
    cmd = [gxx, "-O2", "-DNDEBUG", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM=1", f'-DW4_TORCH_VERSION="{torch.__version__}"',
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           "-I", str(root / "include"), "-I", str(root / "include" / "torch" / "csrc" / "api" / "include"),
           "-I", str(Path(os.environ.get("ROCM_PATH", "/opt/rocm")) / "include"),
           "-I", sysconfig.get_paths()["include"], "-I", str(ROOT / "include"), str(EXT_SRC), "-o", str(tmp),
           "-L", str(root / "lib"), "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10", "-lc10_hip"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed: {EXT_SRC.name}\n{' '.join(cmd)}\n{r.stderr}")
    os.replace(tmp, EXT_LIB)
    return EXT_LIB


def build(jobs: int | None = None, verbose: bool = True) -> Path:
    BUILD.mkdir(exist_ok=True)
    srcs = sources()
    jobs = jobs or min(len(srcs), os.cpu_count() or 4, 8)
    with ThreadPoolExecutor(jobs + 1) as ex:
        ext = ex.submit(build_ext)
        objs = list(ex.map(_compile, srcs))
        ext = ext.result()
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed\n{' '.join(cmd)}\n{r.stderr}")
    os.replace(tmp, LIB)
    bench_srcs = sorted(list(BENCH_SRC.glob("*.hip")) + list(BENCH_SRC.glob("*.cpp")))
    if bench_srcs:
        bobjs = [_compile(s) for s in bench_srcs]
        btmp = BENCH_LIB.with_suffix(".so.tmp")
        cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(btmp), *map(str, bobjs)]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"link failed\n{' '.join(cmd)}\n{r.stderr}")
        os.replace(btmp, BENCH_LIB)
    if verbose:
        more = ", ".join(p.name for p in (ext, BENCH_LIB) if p)
        print(f"built {LIB} from {len(srcs)} sources (+ {more})", file=sys.stderr)
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=None)
    build(ap.parse_args().jobs)
