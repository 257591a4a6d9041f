"""Builds libternary_spmm.so (host packers + gfx950 kernels) with hipcc and _tl_torch.so (the short way from torch calls into
it) with the host compiler, in-tree."""
import os
import shutil
import subprocess
import sysconfig

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG_DIR)
LIB_PATH = os.path.join(PKG_DIR, "libternary_spmm.so")
BINDING_PATH = os.path.join(PKG_DIR, "_tl_torch.so")
SOURCES = ["tl_pack.cpp", "tl_layout.cpp", "tl_kernels.hip", "tl_small_m.hip", "tl_matrix.hip", "tl_few.hip", "tl_decode.hip", "tl_prefill.hip"]


def hipcc():
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found: the gfx950 library cannot be built on this machine")
    return exe


def build_library(verbose=True):
    """Compiles every translation unit for gfx950 and links the shared library. Always recompiles."""
    csrc = os.path.join(PKG_DIR, "csrc")
    cmd = [
        hipcc(), "-shared", "-fPIC", "-O3", "-std=c++17", "--offload-arch=gfx950",
        # packed-fp32 VALU forms are kept out of the generated code
        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
        "-Wall", "-Wno-unused-command-line-argument",
        "-I", os.path.join(ROOT, "include"), "-I", csrc,
        "-x", "hip",
    ] + [os.path.join(csrc, s) for s in SOURCES] + ["-o", LIB_PATH]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    return LIB_PATH


def build_binding(verbose=True):
    """Compiles tl_torch.cpp against the installed torch.  Always recompiles."""
    import torch
    from torch.utils import cpp_extension
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(hipcc())))
    include = cpp_extension.include_paths() + [sysconfig.get_paths()["include"], os.path.join(rocm, "include")]
    cmd = ["g++", "-shared", "-fPIC", "-O2", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           "-D_GLIBCXX_USE_CXX11_ABI=%d" % int(torch._C._GLIBCXX_USE_CXX11_ABI), "-I", os.path.join(ROOT, "include")]
    for path in include:
        cmd += ["-isystem", path]
    cmd += [os.path.join(PKG_DIR, "csrc", "tl_torch.cpp"), "-o", BINDING_PATH]
    cmd += ["-L" + path for path in cpp_extension.library_paths()] + ["-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python"]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    return BINDING_PATH


if __name__ == "__main__":
    build_library()
    build_binding()
