"""Compiles the gfx950 HIP kernels and the C-ABI shim into nexttransformer_amd/_lib/libnt_moe.so, and
the native host path (csrc/host.cpp, a Python module over torch's C++ API) into nt_moe_host.so
beside it.

    python -m nexttransformer_amd.build [-v]

Every translation unit is compiled with hipcc for gfx950 only, in parallel, then linked into one
shared library that the package loads through ctypes. Packed-FP32 instructions are disabled for
all device code (-Xclang -target-feature -Xclang -packed-fp32-ops).
"""
from concurrent.futures import ThreadPoolExecutor
import os
import shutil
import subprocess
import sys
import sysconfig
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
BUILD = PKG / "_build"
LIB = PKG / "_lib" / "libnt_moe.so"
HOST = PKG / "_lib" / "nt_moe_host.so"
ARCH = "gfx950"

FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument", "-Wno-inline-asm",
    f"-I{ROOT / 'include'}", f"-I{CSRC}",
]


def hipcc():
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(path).exists():
        raise RuntimeError("hipcc not found: the MI355X kernels need ROCm's hipcc")
    return path


def sources():
    return sorted(CSRC.glob("*.hip"))


def _compile(src, verbose):
    obj = BUILD / (src.stem + ".o")
    cmd = [hipcc(), *FLAGS, "-c", str(src), "-o", str(obj)]
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{proc.stderr}")
    return obj


def _compile_host(verbose):
    """csrc/host.cpp -> object (host code only, so the host compiler). NDEBUG as torch itself is
    built: without it pybind11's headers put a thread-local counter into the module, and with a
    loaded module's thread-local block never touched, every thread-local access of the process goes
    glibc's slow way (each torch.empty 1.1 -> 1.4 us, a small fp8 forward through the ops 91 -> 101
    us once the module was loaded)."""
    import torch
    from nexttransformer_amd._native import host_marker
    root = Path(torch.__file__).resolve().parent
    obj = BUILD / "host.o"
    cmd = [shutil.which("g++") or "c++", "-O2", "-DNDEBUG", "-std=c++17", "-fPIC", "-fvisibility=hidden",
           f'-DNT_MOE_HOST_MARKER="{host_marker().decode()}"',
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f"-I{ROOT / 'include'}", f"-isystem{root / 'include'}",
           f"-isystem{root / 'include' / 'torch' / 'csrc' / 'api' / 'include'}",
           f"-isystem{sysconfig.get_paths()['include']}", "-c", str(CSRC / "host.cpp"), "-o", str(obj)]
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"the host compiler failed for host.cpp:\n{proc.stderr}")
    return obj, root / "lib"


def _link(cmd, lib, verbose):
    tmp = lib.with_suffix(".so.tmp")
    cmd = [*cmd, "-o", str(tmp)]
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed:\n{proc.stderr}")
    os.replace(tmp, lib)


def build(verbose=False, jobs=None):
    """Compile every source and link libnt_moe.so and nt_moe_host.so; returns the former's path."""
    BUILD.mkdir(parents=True, exist_ok=True)
    LIB.parent.mkdir(parents=True, exist_ok=True)
    srcs = sources()
    jobs = jobs or min(len(srcs) + 1, int(os.environ.get("MAX_JOBS", "8")))
    # the longest compilation first
    srcs.sort(key=lambda p: p.stat().st_size, reverse=True)
    srcs.sort(key=lambda p: p.stem != "grouped_gemm_packed")
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        objs = pool.map(lambda s: _compile(s, verbose), srcs)
        host, torch_lib = pool.submit(_compile_host, verbose).result()
        objs = sorted(map(str, objs))
    _link([hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs], LIB, verbose)
    _link([shutil.which("g++") or "c++", "-shared", str(host), f"-L{torch_lib}", "-lc10",
           "-ltorch_cpu", "-ltorch_python", "-ltorch", f"-L{LIB.parent}", f"-l:{LIB.name}",
           "-Wl,-rpath,$ORIGIN"], HOST, verbose)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
