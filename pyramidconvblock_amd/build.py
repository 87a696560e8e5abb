"""Builds libpdw.so (the C-ABI HIP library) in-tree with hipcc for gfx950.

    python -m pyramidconvblock_amd.build [--force]

Every csrc/*.hip file is compiled to an object (in parallel) and linked into
pyramidconvblock_amd/libpdw.so; csrc/torch_ops.cpp (the operators' host path, no device code) is
compiled with the host compiler against torch's headers and linked to it as the extension module
of ext_path().  hipcc cross-compiles, so no GPU is needed.  libpdw.so needs no torch: run as a script
(python pyramidconvblock_amd/build.py) where there is none, this builds the library alone.
With PDW_TUNE_BUILD=1 in the environment of the build the library is compiled with -DPDW_TUNE, which makes
its planners honour the PDW_* override variables (for experiments; the product build reads no environment).
"""
from __future__ import annotations

import glob
import importlib.util
import os
import re
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "csrc", "build")
LIB = os.path.join(HERE, "libpdw.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = (["-DPDW_TUNE"] if os.environ.get("PDW_TUNE_BUILD") else []) + [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc", "-ffp-contract=fast",
    # keep the compiler from forming packed-fp32 VALU ops
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unknown-warning-option",
]


def _stale(out, deps):
    if not os.path.exists(out):
        return True
    t = os.path.getmtime(out)
    return any(os.path.getmtime(d) > t for d in deps)


def _compile(src, headers, force):
    obj = os.path.join(OBJ, os.path.basename(src)[:-4] + ".o")
    if force or _stale(obj, [src] + headers):
        cmd = [HIPCC] + FLAGS + ["-c", src, "-o", obj]
        r = subprocess.run(cmd, capture_output=True, text=True)
        err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
        if r.returncode != 0:
            raise RuntimeError(f"hipcc failed for {src}:\n{err}")
        if err.strip():
            sys.stderr.write(err + "\n")
    return obj


def ext_path(torch_version: str) -> str:
    """File of the host extension.  It is bound to the interpreter and to the torch it was compiled against, so it
    carries both in its name: after a change of either the file is missing, and is built, instead of being loaded."""
    tag = re.sub(r"[^0-9A-Za-z.]+", "_", f"{sysconfig.get_config_var('SOABI')}-torch{torch_version}")
    return os.path.join(HERE, f"_pdw_torch.{tag}.so")


def _headers():
    return sorted(glob.glob(os.path.join(CSRC, "*.h"))) + [os.path.join(HERE, "..", "include", "pdw.h")]


def build_ext(force: bool = False) -> str:
    """The host extension: libpdw.so is found beside it ($ORIGIN), torch's libraries are loaded by `import torch`."""
    import torch

    src, ext = os.path.join(CSRC, "torch_ops.cpp"), ext_path(torch.__version__)
    if not (force or _stale(ext, [src] + _headers())):
        return ext
    troot = os.path.dirname(torch.__file__)
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall",
           "-D__HIP_PLATFORM_AMD__=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           "-isystem", os.path.join(troot, "include"), "-isystem", os.path.join(troot, "include/torch/csrc/api/include"),
           "-isystem", "/opt/rocm/include", "-isystem", sysconfig.get_paths()["include"], src, "-o", ext,
           LIB, "-L" + os.path.join(troot, "lib"), "-ltorch_python", "-ltorch_cpu", "-ltorch", "-lc10", "-lc10_hip",
           "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"building {os.path.basename(ext)} failed:\n" + r.stderr)
    return ext


def build(force: bool = False, jobs: int | None = None) -> str:
    os.makedirs(OBJ, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    headers = _headers()
    jobs = jobs or min(len(srcs), os.cpu_count() or 4, 16)
    with ThreadPoolExecutor(jobs) as ex:
        objs = list(ex.map(lambda s: _compile(s, headers, force), srcs))
    if force or _stale(LIB, objs):
        cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-fno-gpu-rdc", "-Wl,-soname,libpdw.so", "-o", LIB] + objs
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError("link failed:\n" + r.stderr)
    if importlib.util.find_spec("torch") is None:
        sys.stderr.write("no torch here: libpdw.so is built, the host extension of the Python modules is not\n")
    else:
        build_ext(force)
    return LIB


if __name__ == "__main__":
    print(build(force="--force" in sys.argv))
