"""Build recipe for libmindspeed_amd.so (hipcc, gfx950 only, in-tree).

``python -m mindspeed_amd.build`` compiles every ``csrc/*.hip`` translation
unit for gfx950 and links them into ``mindspeed_amd/libmindspeed_amd.so``,
and builds the native side of the Python ops (``_host.so``) that calls it.
hipcc cross-compiles, so this works on a host without a GPU.
"""
from __future__ import annotations

import hashlib
import os
import re
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ_DIR = os.path.join(HERE, "build")
LIB_PATH = os.path.join(HERE, "libmindspeed_amd.so")
TRACE_LIB_PATH = os.path.join(HERE, "libmindspeed_amd_trace.so")   # diagnostic variant: per-tile time stamps
MICROBENCH_CSRC = os.path.join(HERE, "csrc_microbench")
MICROBENCH_LIB_PATH = os.path.join(HERE, "libmindspeed_amd_microbench.so")   # measurement helpers (plain copy kernel)

HOST_SRC = os.path.join(HERE, "csrc_host", "launch.cpp")
HOST_LIB_PATH = os.path.join(HERE, "_host.so")               # the kernel calls of the Python ops in native code

ARCH = "gfx950"
# packed-fp32 VALU forms are switched off for every device translation unit.
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-fPIC", "-std=c++17",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found: the MI355X kernels cannot be built")
    return exe


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def source_hash() -> str:
    """First 16 hex digits of the SHA-256 over the kernel sources and the native side of the ops (csrc/*.hip, csrc/*.h, the
    C-ABI header, csrc_host/launch.cpp) in name order: names the build that measured figures (profiles/*.json) belong to."""
    h = hashlib.sha256()
    files = sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith((".hip", ".h")))
    files += [os.path.join(HERE, "..", "include", "mindspeed_amd.h"), HOST_SRC]
    for f in files:
        h.update(os.path.basename(f).encode())
        with open(f, "rb") as fh:
            h.update(fh.read())
    return h.hexdigest()[:16]


INTERFACE_HEADERS = (os.path.join(HERE, "..", "include", "mindspeed_amd.h"), os.path.join(CSRC, "internal.h"))


def interface_hash() -> str:
    """First 16 hex digits of the SHA-256 over the declarations of the library's entry points (comments and spacing left
    out).  Compiled into the library and into ``_host.so``, which passes its arguments by these declarations: a pair that
    was not built from the same ones is refused."""
    h = hashlib.sha256()
    for f in INTERFACE_HEADERS:
        with open(f) as fh:
            h.update(" ".join(re.sub(r"/\*.*?\*/|//[^\n]*", " ", fh.read(), flags=re.S).split()).encode())
    return h.hexdigest()[:16]


def _interface_flag() -> str:
    return f'-DMS_INTERFACE="{interface_hash()}"'


def _compile(src: str, force: bool, extra=(), suffix="") -> str:
    obj = os.path.join(OBJ_DIR, os.path.basename(src)[:-4] + suffix + ".o")
    deps = [src, os.path.join(HERE, "..", "include", "mindspeed_amd.h")]
    deps += [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".h")]
    if not force and os.path.exists(obj) and all(os.path.getmtime(obj) > os.path.getmtime(d) for d in deps):
        return obj
    cmd = [_hipcc(), *HIPCC_FLAGS, _interface_flag(), *extra, "-c", src, "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{res.stderr}")
    return obj


def build(force: bool = True, verbose: bool = False) -> str:
    """Compile and link the library; returns its path."""
    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs = sources()
    with ThreadPoolExecutor(max_workers=min(8, len(srcs))) as pool:
        objs = list(pool.map(lambda s: _compile(s, force), srcs))
    cmd = [_hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", LIB_PATH, *objs]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    if verbose:
        print(f"built {LIB_PATH} from {len(srcs)} translation units")
    return LIB_PATH


def compile_trace() -> str:
    """The one translation unit of its own that the diagnostic library has."""
    os.makedirs(OBJ_DIR, exist_ok=True)
    return _compile(os.path.join(CSRC, "gmm_fast.hip"), True, ("-DMS_TRACE_TILES",), "_trace")


def build_trace(verbose: bool = False, force: bool = True) -> str:
    """The diagnostic variant of the library: the bf16 grouped-matmul fast kernels and those of both gradients (one
    translation unit then) compiled with MS_TRACE_TILES (every workgroup records time stamps of its phases, read back with
    ms_trace_read; see profile_tools timeline).  Not loaded by anything else; select it with MINDSPEED_AMD_LIB."""
    os.makedirs(OBJ_DIR, exist_ok=True)
    objs = [_compile(s, force, ("-DMS_TRACE_TILES",), "_trace") if s.endswith("gmm_fast.hip") else _compile(s, False)
            for s in sources() if not s.endswith("gmm_pair.hip")]
    cmd = [_hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", TRACE_LIB_PATH, *objs]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    if verbose:
        print(f"built {TRACE_LIB_PATH}")
    return TRACE_LIB_PATH


def build_microbench(verbose: bool = False) -> str:
    """The measurement helpers (csrc_microbench/*.hip: the plain copy kernel the microbenchmarks and the counter
    calibration use).  A library of its own: nothing in it is part of the product's C ABI."""
    srcs = sorted(os.path.join(MICROBENCH_CSRC, f) for f in os.listdir(MICROBENCH_CSRC) if f.endswith(".hip"))
    cmd = [_hipcc(), *HIPCC_FLAGS, "-shared", "-o", MICROBENCH_LIB_PATH, *srcs]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for the microbench helpers:\n{res.stderr}")
    if verbose:
        print(f"built {MICROBENCH_LIB_PATH}")
    return MICROBENCH_LIB_PATH


def build_host(verbose: bool = False, force: bool = True) -> str:
    """The native side of the Python ops (csrc_host/launch.cpp): host code only, against torch's headers."""
    if not force and os.path.exists(HOST_LIB_PATH) and \
            all(os.path.getmtime(HOST_LIB_PATH) > os.path.getmtime(d) for d in (HOST_SRC, *INTERFACE_HEADERS)):
        return HOST_LIB_PATH
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths, library_paths

    cmd = [os.environ.get("CXX") or "g++", "-O2", "-fPIC", "-shared", "-std=c++17", "-fvisibility=hidden",
           "-DTORCH_EXTENSION_NAME=_host", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           _interface_flag(), "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",      # (the last two: what torch's own stream header asks for)
           *(f"-I{d}" for d in (*include_paths(), sysconfig.get_paths()["include"], "/opt/rocm/include")),
           HOST_SRC, "-o", HOST_LIB_PATH, *(f"-L{d}" for d in library_paths()),
           "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip", "-ltorch_python"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed for {HOST_SRC}:\n{res.stderr}")
    if verbose:
        print(f"built {HOST_LIB_PATH}")
    return HOST_LIB_PATH


def main(args) -> None:
    if "--trace" in args:
        build_trace(verbose=True)
    elif "--microbench" in args:
        build_microbench(verbose=True)
    elif "--host" in args:
        build_host(verbose=True)
    else:                                # the library and what calls it: never one of the two alone
        force = "--incremental" not in args
        with ThreadPoolExecutor(max_workers=1) as pool:
            host = pool.submit(build_host, verbose=True, force=force)
            build(force=force, verbose=True)
            host.result()


if __name__ == "__main__":
    main(sys.argv[1:])
