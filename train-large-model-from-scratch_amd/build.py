"""Build recipe (in-tree outputs): libmoe_gfx950.so, the kernels behind the C ABI (hipcc, gfx950 only),
and _native.so, the autograd nodes on top of it (host C++ against torch)."""
from __future__ import annotations

import os
import subprocess
import sysconfig
from concurrent.futures import ThreadPoolExecutor

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG_DIR, "csrc")
INCLUDE = os.path.join(os.path.dirname(PKG_DIR), "include")
LIB_PATH = os.path.join(PKG_DIR, "libmoe_gfx950.so")
NATIVE_PATH = os.path.join(PKG_DIR, "_native.so")
SOURCES = ("route.hip", "dispatch.hip", "place.hip", "norm.hip", "gemm.hip", "row_ring.hip", "f32.hip", "f32_gemm.hip", "few.hip", "router.hip", "wgrad.hip", "layer.hip")

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # keep the compiler from forming packed-fp32 VALU ops
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.isabs(cand) and os.path.exists(cand) or not os.path.isabs(cand)):
            return cand
    raise RuntimeError("hipcc not found")


def _run(cmd, what, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{what} failed:\n{r.stderr}")


def _native_commands():
    import torch
    from torch.utils import cpp_extension
    obj = os.path.join(CSRC, "binding.o")
    includes = [f"-I{p}" for p in (INCLUDE, CSRC, *cpp_extension.include_paths("cuda"), sysconfig.get_paths()["include"])]
    compile_ = ["g++", "-O2", "-std=c++17", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
                "-DTORCH_EXTENSION_NAME=_native", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
                *includes, "-c", os.path.join(CSRC, "binding.cpp"), "-o", obj]
    libs = [f"-L{p}" for p in cpp_extension.library_paths("cuda")]
    link = ["g++", "-shared", "-o", NATIVE_PATH, obj, *libs, f"-L{PKG_DIR}", "-l:libmoe_gfx950.so", "-lc10", "-lc10_hip",
            "-ltorch_cpu", "-ltorch", "-ltorch_python", "-Wl,-rpath,$ORIGIN"]
    return compile_, link


def build_library(verbose: bool = False) -> str:
    """Compile every source and link both shared libraries.  Always recompiles."""
    objs = [os.path.join(CSRC, src.replace(".hip", ".o")) for src in SOURCES]
    jobs = [([hipcc(), *HIPCC_FLAGS, "-I", INCLUDE, "-I", CSRC, "-c", os.path.join(CSRC, src), "-o", obj],
             f"hipcc on {src}") for src, obj in zip(SOURCES, objs)]
    native_compile, native_link = _native_commands()
    jobs.insert(0, (native_compile, "g++ on binding.cpp"))
    with ThreadPoolExecutor(4) as pool:
        for done in [pool.submit(_run, cmd, what, verbose) for cmd, what in jobs]:
            done.result()
    _run([hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB_PATH, *objs], "link", verbose)
    _run(native_link, "link of _native.so", verbose)
    return LIB_PATH


if __name__ == "__main__":
    print(build_library(verbose=True))
