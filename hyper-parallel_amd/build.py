"""Builds libhpfp8.so (HIP kernels + C ABI) in-tree with hipcc for gfx950, and _native.so (the tensor operators' host path, host
code only) against the installed torch.

Usage: python build.py [--force]
"""
from __future__ import annotations

import importlib.util
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "hpfp8", "libhpfp8.so")
NATIVE = os.path.join(HERE, "hpfp8", "_native.so")
NATIVE_SOURCE = os.path.join(CSRC, "torch_ops.cpp")
SOURCES = ["capi.hip", "quantize.hip", "bucket.hip", "grouped.hip", "gemm.hip", "gemm_skinny.hip"]
HEADERS = ["gemm_skinny.h", "gemm_tile.h", "hpfp8_device.h", "hpfp8_host.h", os.path.join("..", "..", "include", "hpfp8.h")]


def _flags():
    # full IEEE division/sqrt, denormals kept, no packed fp32 arithmetic
    return [
        "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
        "-fno-fast-math", "-ffp-contract=off", "-fno-gpu-flush-denormals-to-zero",
        "-fhip-fp32-correctly-rounded-divide-sqrt",
        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
        # matrix instructions write their results to vector registers also where a kernel could have more of them
        # (4-wave GEMM kernels): through accumulation registers every promotion FMA would need a move
        "-mllvm", "-amdgpu-mfma-vgpr-form",
        "-Wno-unused-command-line-argument",
    ]


def _native_tag() -> str:
    spec = importlib.util.spec_from_file_location("hpfp8_lib", os.path.join(HERE, "hpfp8", "_lib.py"))
    lib = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(lib)
    return lib.native_tag()


def _native_command():
    import torch
    from torch.utils.cpp_extension import include_paths
    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    return (["g++", "-O2", "-std=c++17", "-fPIC", "-shared", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}"]
            + ["-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f'-DHPFP8_BUILT_FOR="{_native_tag()}"']
            + [f"-I{d}" for d in include_paths("cuda") + [sysconfig.get_paths()["include"]]]
            + [NATIVE_SOURCE, "-o", NATIVE, f"-L{lib}", "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip", f"-Wl,-rpath,{lib}"])


def _older(out, deps) -> bool:
    if not os.path.exists(out):
        return True
    t = os.path.getmtime(out)
    return any(os.path.getmtime(d) > t for d in deps + [os.path.abspath(__file__)])


def library_stale() -> bool:
    return _older(OUT, [os.path.join(CSRC, s) for s in SOURCES + HEADERS])


def native_stale() -> bool:
    """Older than its source, or built for another torch or interpreter (the module holds the name of what it was built for)."""
    if _older(NATIVE, [NATIVE_SOURCE, os.path.join(CSRC, HEADERS[-1])]):
        return True
    with open(NATIVE, "rb") as f:
        return _native_tag().encode() + b"\0" not in f.read()


def needs_build() -> bool:
    return library_stale() or native_stale()


def _run(cmd, verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in res.stdout.splitlines() if "packed-fp32-ops" not in l)
    if res.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed:\n" + out)
    if verbose and out.strip():
        print(out)


def build(force: bool = False, verbose: bool = False) -> str:
    """Each of the two where it is stale (``force``: both); the library first, which the package can do with alone."""
    if force or library_stale():
        hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
        _run([hipcc] + _flags() + [os.path.join(CSRC, s) for s in SOURCES] + ["-o", OUT], verbose)
    if force or native_stale():
        _run(_native_command(), verbose)
    return OUT


if __name__ == "__main__":
    print(build(force="--force" in sys.argv, verbose=True))
