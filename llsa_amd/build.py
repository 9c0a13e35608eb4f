"""Builds llsa_amd/lib/libllsa_hip.so from llsa_amd/csrc/*.hip with hipcc for gfx950, and the host module
llsa_amd/lib/_llsa_host.so (the operators' host side and autograd nodes, against torch's headers) with the host compiler.

    python -m llsa_amd.build            # compile every source (parallel), link the two shared libraries

hipcc cross-compiles without a GPU.  The library is kept in-tree (git-ignored) so that a
checkout that was built once can be used on a machine without recompiling.
"""
from __future__ import annotations

import concurrent.futures as cf
import hashlib
import os
import re
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
OBJDIR = os.path.join(HERE, "lib", "obj")
LIBNAME = "libllsa_hip.so"
HOSTNAME = "_llsa_host.so"

HIPCC = os.environ.get("HIPCC") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
CXX = os.environ.get("CXX") or "g++"
ARCH = "gfx950"
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",     # no packed-fp32 VALU ops
    "-mllvm", "-amdgpu-mfma-vgpr-form",      # MFMA results straight into VGPRs: no v_accvgpr copies around the soft-max
    "-Wall", "-Wno-unused-function", "-Wno-unknown-attributes",
]


def sources():
    return sorted(f for f in os.listdir(CSRC) if f.endswith(".hip"))


def kernel_sources_digest() -> str:
    """Names the kernels a measurement was made with: a digest of the device sources without their comments and white space."""
    h = hashlib.sha256()
    for f in sorted(f for f in os.listdir(CSRC) if f.endswith((".hip", ".h"))):
        text = open(os.path.join(CSRC, f)).read()
        text = re.sub(r"/\*.*?\*/", "", re.sub(r"//[^\n]*", "", text), flags=re.S)
        h.update(f.encode() + b"\0" + re.sub(r"\s+", "", text).encode() + b"\0")
    return h.hexdigest()[:16]


def _compile(src: str) -> str:
    obj = os.path.join(OBJDIR, src.replace(".hip", ".o"))
    cmd = [HIPCC, *FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{err}")
    if err.strip():
        print(err, file=sys.stderr)
    return obj


def build_host() -> str:
    """The host module: C++ only, no device code."""
    import sysconfig
    import torch
    base = os.path.dirname(torch.__file__)
    out = os.path.join(LIBDIR, HOSTNAME)
    tmp = out + ".tmp"
    inc = [os.path.join(base, "include"), os.path.join(base, "include", "torch", "csrc", "api", "include"),
           os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"), sysconfig.get_paths()["include"]]
    cmd = [CXX, "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           "-DTORCH_API_INCLUDE_EXTENSION_H", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *(f for d in inc for f in ("-isystem", d)), os.path.join(CSRC, "host", "operators.cpp"), "-o", tmp,
           "-L" + os.path.join(base, "lib"), "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python", "-lamdhip64"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("host module:\n" + r.stderr)
    if r.stderr.strip():
        print(r.stderr, file=sys.stderr)
    os.replace(tmp, out)
    return out


def build(verbose: bool = True) -> str:
    os.makedirs(OBJDIR, exist_ok=True)
    srcs = sources()
    with cf.ThreadPoolExecutor(max_workers=min(8, len(srcs) + 1)) as ex:
        host = ex.submit(build_host)
        objs = list(ex.map(_compile, srcs))
        host.result()
    out = os.path.join(LIBDIR, LIBNAME)
    tmp = out + ".tmp"
    r = subprocess.run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stderr)
    os.replace(tmp, out)
    if verbose:
        print(f"built {out} from {len(srcs)} sources, and {HOSTNAME}")
    return out


if __name__ == "__main__":
    build()
