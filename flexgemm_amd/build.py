"""Build recipe of libflexgemm_hip.so: hipcc, gfx950 only, in-tree output.

`python -m flexgemm_amd.build` compiles every file under flexgemm_amd/csrc/ and links
flexgemm_amd/_lib/libflexgemm_hip.so, then the tests' torch-free caller of the C ABI against it
(flexgemm_amd/_lib/conv_host).  Objects are rebuilt when their source (or a header) is newer; pass
--force to rebuild everything.
"""
from __future__ import annotations

import glob
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

PKG = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG, "csrc")
OUT_DIR = os.path.join(PKG, "_lib")
LIB = os.path.join(OUT_DIR, "libflexgemm_hip.so")
# the operators' host side: a Python extension over torch's C++ API (host code only: no kernels in it)
HOST_SRC = os.path.join(CSRC, "host", "fgx_host.cpp")
HOST_LIB = os.path.join(OUT_DIR, "fgx_host.so")
# a caller of the C ABI without Python or torch, run by the GPU tests (tests/cabi_host/conv_host.cpp)
HOST_CHECK_SRC = os.path.join(PKG, "..", "tests", "cabi_host", "conv_host.cpp")
HOST_CHECK = os.path.join(OUT_DIR, "conv_host")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

COMMON_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unknown-warning-option",
    "-DNDEBUG",
]


def _headers():
    return glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(PKG, "..", "include", "*.h"))


def _stale(target: str, deps) -> bool:
    if not os.path.exists(target):
        return True
    t = os.path.getmtime(target)
    return any(os.path.getmtime(d) > t for d in deps)


def _host_command():
    import sysconfig
    import torch
    from torch.utils import cpp_extension
    includes = cpp_extension.include_paths() + [sysconfig.get_paths()["include"], "/opt/rocm/include"]
    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    return (["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall", "-Wno-unknown-pragmas", "-D__HIP_PLATFORM_AMD__",
             f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-DTORCH_EXTENSION_NAME=fgx_host", "-DNDEBUG"]
            + [f for i in includes for f in ("-isystem", i)]
            + [HOST_SRC, "-o", HOST_LIB, "-L", torch_lib, "-lc10", "-lc10_hip", "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lamdhip64", "-ldl"])


def build(force: bool = False, verbose: bool = True, jobs: int = 4) -> str:
    os.makedirs(OUT_DIR, exist_ok=True)
    sources = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    if not sources:
        raise RuntimeError("no HIP sources found under " + CSRC)
    hdrs = _headers()
    objs = []
    todo = []
    for src in sources:
        obj = os.path.join(OUT_DIR, os.path.basename(src)[:-4] + ".o")
        objs.append(obj)
        if force or _stale(obj, [src] + hdrs):
            todo.append((src, obj))

    def compile_one(item):
        src, obj = item
        cmd = [HIPCC] + COMMON_FLAGS + ["-c", src, "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src}:\n{r.stdout}\n{r.stderr}")
        warn = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l and l.strip())
        if verbose and warn:
            print(warn, flush=True)

    def compile_host():
        cmd = _host_command()
        if verbose:
            print(" ".join(cmd), flush=True)
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"g++ failed on {HOST_SRC}:\n{r.stdout}\n{r.stderr}")

    with ThreadPoolExecutor(max_workers=max(1, jobs)) as ex:
        host = ex.submit(compile_host) if force or _stale(HOST_LIB, [HOST_SRC] + hdrs) else None
        list(ex.map(compile_one, todo))
        if host is not None:
            host.result()
    if force or todo or _stale(LIB, objs):
        cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-fno-gpu-rdc"] + objs + ["-o", LIB]
        if verbose:
            print(" ".join(cmd), flush=True)
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    if os.path.exists(HOST_CHECK_SRC) and (force or todo or _stale(HOST_CHECK, [HOST_CHECK_SRC, LIB] + hdrs)):
        cmd = [HIPCC] + COMMON_FLAGS + ["-I", os.path.join(PKG, "..", "include"), HOST_CHECK_SRC, "-L", OUT_DIR, "-lflexgemm_hip",
                                        "-Wl,-rpath,$ORIGIN", "-o", HOST_CHECK]
        if verbose:
            print(" ".join(cmd), flush=True)
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"building the host check failed:\n{r.stdout}\n{r.stderr}")
    return LIB


if __name__ == "__main__":
    print(build(force="--force" in sys.argv))
