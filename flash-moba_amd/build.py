"""Builds libflash_moba_hip.so (the C-ABI kernel library) for gfx950 with hipcc.

    python flash-moba_amd/build.py            # build into flash-moba_amd/lib/

hipcc cross-compiles for gfx950 without a GPU.  The library is built in-tree so that it
travels with the source tree; nothing is installed into site-packages.
"""
import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIBDIR, "libflash_moba_hip.so")
HOST_MODULE = "flash_moba_host"  # the eager host path (csrc/torch_ops.cpp), a Python extension beside the library
HOST_LIB = os.path.join(LIBDIR, HOST_MODULE + ".so")
SOURCES = ["fmoba_host.hip", "mean_pool.hip", "topk_csc.hip", "varlen_sort.hip", "attn_fwd.hip", "attn_fwd_rows.hip", "attn_fwd_rows_wide.hip", "attn_fwd_few.hip", "attn_bwd.hip", "attn_bwd_wide.hip"]
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # keep packed-fp32 VALU ops out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


# The compiler's choice between ordinary and accumulation registers for the results of matrix products, for kernels of 512 registers whose
# results vector instructions read: left to itself it takes accumulation registers for all of them and copies (attn_fwd_rows_wide.hip: 600 copies
# in the loop of 64 products, 60 with the flag).
FILE_FLAGS = {"attn_fwd_rows_wide.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"]}


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (looked at $HIPCC, /opt/rocm/bin/hipcc and PATH)")


def _compile(src: str, objdir: str) -> str:
    obj = os.path.join(objdir, src.replace(".hip", ".o"))
    cmd = [hipcc()] + FLAGS + FILE_FLAGS.get(src, []) + ["-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("hipcc failed for %s:\n%s\n%s" % (src, r.stdout, r.stderr))
    return obj


def _run(cmd, what):
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("%s failed:\n%s\n%s" % (what, r.stdout, r.stderr))


def _compile_host_module(objdir: str) -> str:
    """torch_ops.cpp against the installed torch (host code only: the host compiler)."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths

    inc = include_paths() + [os.path.join(os.path.dirname(os.path.dirname(hipcc())), "include"), sysconfig.get_paths()["include"]]
    obj = os.path.join(objdir, "torch_ops.o")
    _run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
          "-DTORCH_EXTENSION_NAME=" + HOST_MODULE, "-D_GLIBCXX_USE_CXX11_ABI=%d" % int(torch._C._GLIBCXX_USE_CXX11_ABI)]
         + ["-isystem" + d for d in inc] + ["-c", os.path.join(CSRC, "torch_ops.cpp"), "-o", obj], "compiling the host module")
    return obj


def _link_host_module(obj: str) -> None:
    from torch.utils.cpp_extension import library_paths

    tmp = HOST_LIB + ".tmp"
    _run([os.environ.get("CXX", "g++"), "-shared", "-o", tmp, obj, "-L" + LIBDIR, "-lflash_moba_hip", "-Wl,-rpath,$ORIGIN"]
         + ["-L" + d for d in library_paths()] + ["-l" + x for x in ("torch", "torch_cpu", "torch_hip", "torch_python", "c10", "c10_hip")],
         "linking the host module")
    os.replace(tmp, HOST_LIB)


def build_library(verbose: bool = True, jobs: int = 6) -> str:
    objdir = os.path.join(HERE, "build")
    os.makedirs(objdir, exist_ok=True)
    os.makedirs(LIBDIR, exist_ok=True)
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        host = ex.submit(_compile_host_module, objdir)
        objs = list(ex.map(lambda s: _compile(s, objdir), SOURCES))
    tmp = LIB + ".tmp"
    cmd = [hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n%s\n%s" % (r.stdout, r.stderr))
    os.replace(tmp, LIB)
    _link_host_module(host.result())
    if verbose:
        print("built", LIB, os.path.getsize(LIB), "bytes")
    return LIB


if __name__ == "__main__":
    build_library()
    sys.exit(0)
