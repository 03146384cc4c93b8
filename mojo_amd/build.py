"""Compile the HIP sources under ``mojo_amd/csrc`` into ``mojo_amd/libqmm.so``.

Explicit ``hipcc`` lines for gfx950: one object per source file (compiled side by side), then one
link.  Nothing is built at import time.
"""
from __future__ import annotations

import glob
import os
import subprocess
import sys
import warnings
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
LIB = os.path.join(HERE, "libqmm.so")
CALL = os.path.join(HERE, "_call.so")  # the extension module in front of libqmm.so

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "-O3",
    "-std=c++17",
    "--offload-arch=gfx950",
    "-fPIC",
    # quantisers are specified as separate IEEE operations; hot loops call fmaf explicitly
    "-ffp-contract=off",
    # no compiler-generated packed fp32 arithmetic
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
]


# Per-file additions.  Kernel-argument preloading (the first dwords of the argument block arrive in scalar registers
# with the wavefront instead of through a scalar load) for the kernels whose first microsecond decides a launch.
PER_FILE_FLAGS = {
    "gemv_q4k_lanes.hip": ["-mllvm", "-amdgpu-kernarg-preload-count=12"],
    "gemv_kquant_small.hip": ["-mllvm", "-amdgpu-kernarg-preload-count=12"],
    "gemv_gptq_small.hip": ["-mllvm", "-amdgpu-kernarg-preload-count=14"],
    "gemm_q4_0.hip": ["-mllvm", "-amdgpu-kernarg-preload-count=14"],
    "gemv_q4_0.hip": ["-mllvm", "-amdgpu-kernarg-preload-count=14"],
    "gemm_direct.hip": ["-mllvm", "-amdgpu-kernarg-preload-count=14"],
    "gemm_shared.hip": ["-mllvm", "-amdgpu-kernarg-preload-count=14"],
    "gemm_staged.hip": ["-mllvm", "-amdgpu-kernarg-preload-count=14"],
}


def sources() -> list[str]:
    return sorted(glob.glob(os.path.join(CSRC, "*.hip")))


def _headers_mtime() -> float:
    hdrs = glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(HERE, "..", "include", "*.h"))
    return max(os.path.getmtime(h) for h in hdrs)


def _compile(src: str, obj: str, verbose: bool) -> None:
    cmd = [HIPCC, *FLAGS, *PER_FILE_FLAGS.get(os.path.basename(src), []), "-c", "-o", obj, src]
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        sys.stderr.write(proc.stdout + proc.stderr)
        raise RuntimeError(f"hipcc failed on {os.path.basename(src)}")
    noise = "not a recognized feature for this target"  # the host pass does not know the gfx950 feature flag
    rest = [ln for ln in proc.stderr.splitlines() if ln.strip() and noise not in ln]
    if verbose and rest:
        sys.stderr.write("\n".join(rest) + "\n")


def build(verbose: bool = False, force: bool = True, jobs: int | None = None) -> str:
    """Compile every source (``force=False``: only those newer than their object) and link the library."""
    os.makedirs(OBJ, exist_ok=True)
    hdr_time = _headers_mtime()
    todo, objs = [], []
    for src in sources():
        obj = os.path.join(OBJ, os.path.basename(src)[:-4] + ".o")
        objs.append(obj)
        if force or not os.path.exists(obj) or os.path.getmtime(obj) < max(os.path.getmtime(src), hdr_time):
            todo.append((src, obj))
    jobs = jobs or min(8, os.cpu_count() or 1)
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        for fut in [pool.submit(_compile, s, o, verbose) for s, o in todo]:
            fut.result()
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, *objs]
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        sys.stderr.write(proc.stdout + proc.stderr)
        raise RuntimeError("hipcc failed linking libqmm.so")
    _build_call(force, verbose)
    return LIB


def _build_call(force: bool, verbose: bool) -> None:
    """The extension module ``_call`` (host code only) against the headers of the installed torch and ``libqmm.so``.

    The package works without it (through ctypes), so where it cannot be compiled that is a warning, and no older module stays."""
    from . import _lib

    src = os.path.join(CSRC, "py_call.cpp")
    if not force and _lib.call_is_current(CALL) and os.path.getmtime(CALL) > max(os.path.getmtime(src), _headers_mtime()):
        return
    import sysconfig

    import torch

    root = os.path.dirname(torch.__file__)
    cmd = [HIPCC, "-O2", "-std=c++17", "-fPIC", "-shared", "-x", "c++", "-DUSE_ROCM", "-D__HIP_PLATFORM_AMD__=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f'-DQMM_CALL_STAMP="{_lib.call_stamp()}"', f"-I{root}/include", f"-I{root}/include/torch/csrc/api/include", f"-I{sysconfig.get_paths()['include']}",
           f"-I{os.path.join(os.path.dirname(os.path.dirname(HIPCC)), 'include')}", src,
           "-o", CALL, f"-L{HERE}", "-l:libqmm.so", f"-L{root}/lib", "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip", "-Wl,-rpath,$ORIGIN"]
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        sys.stderr.write(proc.stdout + proc.stderr)
        if os.path.exists(CALL):
            os.remove(CALL)
        warnings.warn("hipcc failed on py_call.cpp: calls will go through ctypes", RuntimeWarning)


if __name__ == "__main__":
    build(verbose=True, force="--incremental" not in sys.argv)
