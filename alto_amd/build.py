"""Builds libalto_mxfp4.so (hand-written HIP for gfx950, hipcc) and alto_mxfp4_host.so (the native host side, g++) in-tree.

Usage: ``python -m alto_amd.build [--force]``.  The library lands in ``alto_amd/lib/`` next to the
sources so that it travels with the tree; nothing is installed outside the repository.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
OBJDIR = os.path.join(HERE, "lib", "obj")
LIBNAME = "libalto_mxfp4.so"
HOSTNAME = "alto_mxfp4_host.so"   # CPython module of csrc/host.cpp, named as its PYBIND11_MODULE
HOSTSRC = os.path.join(CSRC, "host.cpp")
HEADER = os.path.join(HERE, "..", "include", "alto_mxfp4.h")

SOURCES = ["capi.hip", "quantize.hip", "dequantize.hip", "gemm.hip", "gemm_tiled.hip", "gemm_mid.hip", "gemm_skinny.hip", "grouped_gemm.hip", "probe.hip", "qdq.hip", "attention.hip", "attention_split.hip", "attention_quantize.hip", "quantize_dynamic.hip", "random.hip"]

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-gpu-rdc",
    # packed-FP32 VALU forms are kept out of the generated code on purpose
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]

HOST_FLAGS = ["-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1"]


def lib_path() -> str:
    return os.path.join(LIBDIR, LIBNAME)


def host_path() -> str:
    return os.path.join(LIBDIR, HOSTNAME)


def stamp_path(path: str = "") -> str:
    return (path or lib_path()) + ".srchash"


def _digest(first: str, files) -> str:
    import hashlib
    h = hashlib.sha256(first.encode())
    for f in files:
        h.update(os.path.basename(f).encode())
        with open(f, "rb") as fh:
            h.update(fh.read())
    return h.hexdigest()


def source_hash() -> str:
    """Digest of every file the library is built from (kernels, their headers, the C ABI header, the compiler flags)."""
    files = sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith((".hip", ".h")))
    return _digest(" ".join(HIPCC_FLAGS), files + [HEADER])


def host_hash() -> str:
    """Digest of what the host module is built from: its source, the C ABI header whose functions it calls, the flags, and the
    interpreter and torch whose binary interfaces it is compiled against."""
    import torch
    return _digest(" ".join([*HOST_FLAGS, sys.implementation.cache_tag, torch.__version__, str(torch._C._GLIBCXX_USE_CXX11_ABI)]), [HOSTSRC, HEADER])


def _recorded(path: str) -> str:
    try:
        with open(stamp_path(path)) as f:
            return f.read().strip()
    except OSError:
        return ""


def is_stale() -> bool:
    """True when the built library does not come from the sources in the tree (or carries no record of its sources)."""
    return _recorded(lib_path()) != source_hash()


def host_is_stale() -> bool:
    """True when there is no host module, or one of other sources, another interpreter or another torch than these."""
    return not os.path.exists(host_path()) or _recorded(host_path()) != host_hash()


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found: the MXFP4 kernels need the ROCm toolchain to build")
    return exe


def _rocm_include() -> str:
    """Where the HIP runtime's headers are (torch's stream header names its types)."""
    return os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(_hipcc()))), "include")


def _compile(src: str) -> str:
    obj = os.path.join(OBJDIR, os.path.splitext(src)[0] + ".o")
    cmd = [_hipcc(), *HIPCC_FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{res.stdout}\n{res.stderr}")
    return obj


def build_host() -> str:
    """Compile csrc/host.cpp against the installed torch: host code only, so the host compiler does it."""
    import sysconfig

    import torch
    os.makedirs(LIBDIR, exist_ok=True)
    digest = host_hash()
    tdir = os.path.dirname(torch.__file__)
    out = host_path()
    tmp = f"{out}.{os.getpid()}.tmp"
    cmd = [shutil.which("g++") or "g++", *HOST_FLAGS, f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f"-I{tdir}/include",
           f"-I{tdir}/include/torch/csrc/api/include", f"-I{sysconfig.get_paths()['include']}", f"-I{_rocm_include()}", HOSTSRC, "-o", tmp, f"-L{tdir}/lib",
           "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed for host.cpp:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, out)
    with open(stamp_path(out), "w") as f:
        f.write(digest + "\n")
    return out


def build(verbose: bool = True) -> str:
    """Compile every HIP source, link the shared library and build the host module; always rebuilds."""
    os.makedirs(OBJDIR, exist_ok=True)
    digest = source_hash()   # taken before compiling: an edit made during the build leaves the library marked stale
    with ThreadPoolExecutor(max_workers=min(8, len(SOURCES))) as pool:
        host = pool.submit(build_host)
        objs = list(pool.map(_compile, SOURCES))
        host.result()
    out = lib_path()
    tmp = out + ".tmp"
    cmd = [_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, out)
    with open(stamp_path(), "w") as f:
        f.write(digest + "\n")
    if verbose:
        print(f"built {out} ({os.path.getsize(out)} bytes)")
    return out


if __name__ == "__main__":
    build()
    sys.exit(0)
