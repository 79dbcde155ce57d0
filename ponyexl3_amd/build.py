"""Builds libexl3_hip.so (gfx950) in-tree with hipcc.

``python -m ponyexl3_amd.build`` or ``ponyexl3_amd.build.build()``. Each .hip
file is one translation unit compiled in parallel; the objects are linked into
``ponyexl3_amd/libexl3_hip.so``, the C-ABI library declared in
``include/exl3_hip.h``, and (``diag.hip`` alone) ``ponyexl3_amd/libexl3_diag.so``,
the measurement probes declared in ``include/exl3_diag.h``. ``torch_host.cpp``, the
modules' host path over that library, becomes ``ponyexl3_amd/_exl3_host.so``.
"""

from __future__ import annotations

import concurrent.futures
import os
import shutil
import subprocess
import sys
import sysconfig

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG_DIR, "csrc")
OBJ_DIR = os.path.join(CSRC, "build")
LIB_PATH = os.path.join(PKG_DIR, "libexl3_hip.so")

SOURCES = ["decode.hip", "hadamard.hip", "gemv.hip", "linear_batch.hip", "linear_mid.hip", "linear_rows.hip", "gemm.hip", "moe.hip", "moe_route.hip", "moe_rows.hip", "search.hip", "capi.hip"]
# measurement probes (include/exl3_diag.h): a library of their own, kept out of the product ABI
DIAG_SOURCES = ["diag.hip"]
DIAG_LIB_PATH = os.path.join(PKG_DIR, "libexl3_diag.so")

HOST_SOURCE = "torch_host.cpp"
HOST_LIB_PATH = os.path.join(PKG_DIR, "_exl3_host.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fvisibility=hidden",
    "-Wall",
    "-Wno-unused-function",
    # packed fp32 VALU ops are kept out of the generated code on this hardware pool
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; the EXL3 kernels need the ROCm toolchain")
    return exe


def _compile(src: str, extra: list[str]) -> str:
    obj = os.path.join(OBJ_DIR, os.path.splitext(src)[0] + ".o")
    cmd = [hipcc(), *HIPCC_FLAGS, *extra, "-c", os.path.join(CSRC, src), "-o", obj]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{proc.stderr[-8000:]}")
    noise = "packed-fp32-ops"  # host pass does not know -packed-fp32-ops; harmless
    warn = "\n".join(l for l in proc.stderr.splitlines() if noise not in l and l.strip())
    if warn:
        sys.stderr.write(warn + "\n")
    return obj


def _compile_host() -> str:
    """The CPython extension against this interpreter's torch; returns its object file."""
    import torch

    inc = os.path.join(os.path.dirname(torch.__file__), "include")
    obj = os.path.join(OBJ_DIR, "torch_host.o")
    abi = int(torch._C._GLIBCXX_USE_CXX11_ABI)
    cmd = [shutil.which("g++") or "c++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-Wall",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={abi}",
           "-isystem", inc, "-isystem", os.path.join(inc, "torch", "csrc", "api", "include"),
           "-isystem", os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"),
           "-isystem", sysconfig.get_paths()["include"],
           "-c", os.path.join(CSRC, HOST_SOURCE), "-o", obj]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"g++ failed for {HOST_SOURCE}:\n{proc.stderr[-8000:]}")
    if proc.stderr.strip():
        sys.stderr.write(proc.stderr)
    return obj


def _link_host(obj: str) -> None:
    import torch

    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    cmd = [shutil.which("g++") or "c++", "-shared", "-o", HOST_LIB_PATH, obj, f"-L{lib}", f"-L{PKG_DIR}",
           "-lexl3_hip", "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python", "-Wl,-rpath,$ORIGIN"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed:\n{proc.stderr[-4000:]}")


def build(verbose: bool = False, jobs: int | None = None, extra_flags: list[str] | None = None) -> str:
    os.makedirs(OBJ_DIR, exist_ok=True)
    extra = list(extra_flags or [])
    every = SOURCES + DIAG_SOURCES
    jobs = jobs or min(len(every) + 1, int(os.environ.get("MAX_JOBS", "8")))
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as pool:
        host = pool.submit(_compile_host)
        objs = list(pool.map(lambda s: _compile(s, extra), every))
    for path, group in ((LIB_PATH, objs[: len(SOURCES)]), (DIAG_LIB_PATH, objs[len(SOURCES):])):
        cmd = [hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", path, *group]
        proc = subprocess.run(cmd, capture_output=True, text=True)
        if proc.returncode != 0:
            raise RuntimeError(f"link failed:\n{proc.stderr[-4000:]}")
        if verbose:
            print(f"built {path} ({os.path.getsize(path)} bytes)")
    _link_host(host.result())
    if verbose:
        print(f"built {HOST_LIB_PATH} ({os.path.getsize(HOST_LIB_PATH)} bytes)")
    return LIB_PATH


if __name__ == "__main__":
    build(verbose=True)
