"""Build libt2t_attn.so (HIP, gfx950) and _t2t_host.so (its torch host side,
C++) in-tree.

    python -m tagseq2tagseq_amd.build

Compiles every ``csrc/*.hip`` to an object and links one shared library next
to this file, and ``csrc/host_ops.cpp`` to an extension module that links to
it.  Always recompiles (the build is the "does it compile" check).
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libt2t_attn.so")
HOST = os.path.join(HERE, "_t2t_host.so")
ARCH = os.environ.get("T2T_OFFLOAD_ARCH", "gfx950")

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-munsafe-fp-atomics",
    # Packed-FP32 VALU forms are kept out of the device code.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
]


def _hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(path):
        raise RuntimeError("hipcc not found; the HIP toolchain is required to build libt2t_attn.so")
    return path


def _compile(src: str) -> str:
    obj = os.path.join(OBJ, os.path.basename(src).replace(".hip", ".o"))
    cmd = [_hipcc(), *HIPCC_FLAGS, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr}")
    return obj


def _compile_host() -> str:
    """csrc/host_ops.cpp against this Python and torch (no device code)."""
    import torch
    import sysconfig
    from torch.utils import cpp_extension
    obj = os.path.join(OBJ, "host_ops.o")
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(_hipcc())))
    inc = [*cpp_extension.include_paths(), sysconfig.get_paths()["include"],
           os.path.join(rocm, "include")]
    cmd = [shutil.which("g++") or "c++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_EXTENSION_NAME=_t2t_host",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
           *[f"-I{d}" for d in inc], "-c", os.path.join(CSRC, "host_ops.cpp"), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed for host_ops.cpp:\n{r.stderr[-4000:]}")
    return obj


def _link_host(obj: str) -> None:
    from torch.utils import cpp_extension
    tmp = HOST + ".tmp"
    cmd = [shutil.which("g++") or "c++", "-shared", "-o", tmp, obj, f"-L{HERE}", "-l:libt2t_attn.so",
           "-Wl,-rpath,$ORIGIN", *[f"-L{d}" for d in cpp_extension.library_paths()],
           "-ltorch_python", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(tmp, HOST)


def build(verbose: bool = False) -> str:
    os.makedirs(OBJ, exist_ok=True)
    srcs = sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))
    with ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        host = ex.submit(_compile_host)
        objs = list(ex.map(_compile, srcs))
        host_obj = host.result()
    tmp = LIB + ".tmp"
    cmd = [_hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(tmp, LIB)
    _link_host(host_obj)
    if verbose:
        print(f"built {LIB}")
        print(f"built {HOST}")
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
