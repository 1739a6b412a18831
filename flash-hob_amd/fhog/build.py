"""Build libfhog_hip.so (gfx950) and _fhog_torch.so in-tree.

The shared library holds the HIP kernels and the C ABI declared in ``include/fhog_hip.h``; the extension module is the
native host side of the PyTorch entry points on top of that ABI.  Both are compiled ahead of time (hipcc cross-compiles
without a GPU); nothing is JIT-compiled at run time.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent            # .../flash-hob_amd/fhog
CSRC = PKG_DIR.parent / "csrc"
INCLUDE = PKG_DIR.parent.parent / "include"
LIB_PATH = PKG_DIR / "libfhog_hip.so"
SOURCES = ["fhog_abi.hip", "fhog_rowdot.hip", "fhog_split.hip", "fhog_split_few.hip", "fhog_bf16.hip", "fhog_bf16_pc.hip", "fhog_bf16_ddo.hip", "fhog_small.hip", "fhog_attn.hip", "fhog_attn_split.hip", "fhog_probe.hip"]

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-gpu-rdc",
    # packed-fp32 VALU forms are kept out of every kernel of this library
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # registers spill to scratch memory only: this compiler (clang 22.0.0git, roc-7.2.0) loses registers that it spills to AGPRs
    # out of a tuple that it reloads into AGPRs. In the sweep for dK2 and dV2 of fp16 tensors at d = 128 (split products, two waves
    # on the same rows, band mask) v[8:11] goes to scratch (v8 to v10) and a189 (v11); a[64:67], an operand of the next MFMAs,
    # comes back as three registers from scratch, a189 is never read and a67 still holds an accumulator: NaN in dK2.
    # Of the other files only fhog_attn_split.hip has code that differs with the flag.
    "-mllvm", "-amdgpu-spill-vgpr-to-agpr=0",
    "-Wno-unused-command-line-argument",
] + os.environ.get("FHOG_EXTRA", "").split()   # extra hipcc flags for experiments


def hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; libfhog_hip.so cannot be built")
    return exe


def _torch_ext_commands(obj: Path):
    """g++ command lines that compile csrc/fhog_torch.cpp and link it against torch and libfhog_hip.so next to it."""
    import torch
    from torch.utils.cpp_extension import include_paths, library_paths
    inc = [f"-I{p}" for p in (*include_paths("cuda"), sysconfig.get_paths()["include"], INCLUDE)]
    compile_ = ["g++", "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_EXTENSION_NAME=_fhog_torch",
                f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *inc, "-c", str(CSRC / "fhog_torch.cpp"), "-o", str(obj)]
    link = ["g++", "-shared", "-o", str(PKG_DIR / "_fhog_torch.so"), str(obj), *(f"-L{p}" for p in library_paths("cuda")), f"-L{PKG_DIR}",
            "-lc10", "-lc10_hip", "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lfhog_hip", "-Wl,-rpath,$ORIGIN"]
    return compile_, link


def build(verbose: bool = True, jobs: int = 10) -> Path:
    """Compile every source and link ``libfhog_hip.so`` and ``_fhog_torch.so`` next to this file. Always recompiles."""
    objdir = PKG_DIR.parent / "build"
    objdir.mkdir(exist_ok=True)
    procs = []
    objs = []
    for src in SOURCES:
        obj = objdir / (src + ".o")
        objs.append(str(obj))
        cmd = [hipcc(), *HIPCC_FLAGS, f"-I{INCLUDE}", f"-I{CSRC}", "-c", str(CSRC / src), "-o", str(obj)]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
        if len(procs) >= jobs:
            _drain(procs, verbose)
    ext_obj = objdir / "fhog_torch.o"
    ext_compile, ext_link = _torch_ext_commands(ext_obj)
    if verbose:
        print(" ".join(ext_compile), flush=True)
    procs.append(("fhog_torch.cpp", subprocess.Popen(ext_compile, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
    _drain(procs, verbose)
    cmd = [hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(LIB_PATH), *objs]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    if verbose:
        print(" ".join(ext_link), flush=True)
    subprocess.run(ext_link, check=True)
    return LIB_PATH


def _drain(procs, verbose):
    for src, pr in procs:
        out, _ = pr.communicate()
        lines = [l for l in out.splitlines() if "packed-fp32-ops" not in l]
        if pr.returncode != 0:
            raise RuntimeError(f"compiling {src} failed:\n" + "\n".join(lines))
        if verbose and lines:
            print("\n".join(lines), flush=True)
    procs.clear()


if __name__ == "__main__":
    build()
    print("built", LIB_PATH)
    sys.exit(0)
