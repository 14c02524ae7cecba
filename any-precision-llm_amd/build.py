"""Builds the in-tree native libraries of this package.

    python build.py            # libanyprec_hip.so (hipcc, gfx950), the torch module over it and the host-check lib (g++)

The HIP library is cross-compiled; no GPU is needed to build it.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
OBJDIR = os.path.join(HERE, "build")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")

HIP_LIB = os.path.join(LIBDIR, "libanyprec_hip.so")
TORCH_MODULE = os.path.join(LIBDIR, "_anyprec_torch.so")
HOSTCHECK_LIB = os.path.join(LIBDIR, "libanyprec_hostcheck.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-fno-gpu-rdc",
    "-Wall", "-Wno-unused-function",
]


def _hipcc() -> str:
    for cand in (shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found")


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    # the host pass does not know the packed-fp32 feature and says so; drop that line
    out = "\n".join(l for l in res.stdout.splitlines() if "packed-fp32-ops" not in l)
    if res.returncode != 0:
        raise RuntimeError("command failed: " + " ".join(cmd) + "\n" + out)
    if verbose and out.strip():
        print(out)


def build_hip(verbose: bool = False, extra_flags=(), jobs: int = 8) -> str:
    """One object per kernel family and bit-width (compiled in parallel) + the C ABI, linked into the .so."""
    from concurrent.futures import ThreadPoolExecutor

    os.makedirs(OBJDIR, exist_ok=True)
    os.makedirs(LIBDIR, exist_ok=True)
    compile_flags = [f for f in HIPCC_FLAGS if f != "-shared"] + list(extra_flags) + ["-I", INCLUDE, "-I", CSRC, "-c"]
    units = [(os.path.join(CSRC, "ap_capi.hip"), os.path.join(OBJDIR, "ap_capi.o"), [])]
    for b in range(3, 9):
        units.append((os.path.join(CSRC, "ap_gemv_inst.hip"), os.path.join(OBJDIR, f"ap_gemv_b{b}.o"), [f"-DAP_BITS={b}"]))
        units.append((os.path.join(CSRC, "ap_gemvf_inst.hip"), os.path.join(OBJDIR, f"ap_gemvf_b{b}.o"), [f"-DAP_BITS={b}"]))
        units.append((os.path.join(CSRC, "ap_gemvp_inst.hip"), os.path.join(OBJDIR, f"ap_gemvp_b{b}.o"), [f"-DAP_BITS={b}"]))
        units.append((os.path.join(CSRC, "ap_gemm_inst.hip"), os.path.join(OBJDIR, f"ap_gemm_b{b}.o"), [f"-DAP_BITS={b}"]))
        units.append((os.path.join(CSRC, "ap_gemmw_inst.hip"), os.path.join(OBJDIR, f"ap_gemmw_b{b}.o"), [f"-DAP_BITS={b}"]))
        units.append((os.path.join(CSRC, "ap_gemmt_inst.hip"), os.path.join(OBJDIR, f"ap_gemmt_b{b}.o"), [f"-DAP_BITS={b}"]))
        units.append((os.path.join(CSRC, "ap_gemmb_inst.hip"), os.path.join(OBJDIR, f"ap_gemmb_b{b}.o"), [f"-DAP_BITS={b}"]))
        units.append((os.path.join(CSRC, "ap_gemms_inst.hip"), os.path.join(OBJDIR, f"ap_gemms_b{b}.o"), [f"-DAP_BITS={b}"]))
        units.append((os.path.join(CSRC, "ap_gemv4_inst.hip"), os.path.join(OBJDIR, f"ap_gemv4_b{b}.o"), [f"-DAP_BITS={b}"]))
    hipcc = _hipcc()
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        list(pool.map(lambda u: _run([hipcc, *compile_flags, *u[2], u[0], "-o", u[1]], verbose), units))
    _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-fno-gpu-rdc", *[u[1] for u in units], "-o", HIP_LIB],
         verbose)
    return HIP_LIB


def build_torch(verbose: bool = False) -> str:
    """The Python module over libanyprec_hip.so (host code only).  torch's libraries are found by name: whoever imports the
    module has imported torch before."""
    import sysconfig

    import torch
    torch_dir = os.path.dirname(torch.__file__)
    include = os.path.join(torch_dir, "include")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f'-DAP_TORCH_VERSION="{torch.__version__}"', "-I", INCLUDE, "-isystem", include,
           "-isystem", os.path.join(include, "torch", "csrc", "api", "include"), "-isystem", "/opt/rocm/include",
           "-isystem", sysconfig.get_paths()["include"], os.path.join(CSRC, "ap_torch.cpp"), "-o", TORCH_MODULE,
           "-L", LIBDIR, "-lanyprec_hip", "-L", os.path.join(torch_dir, "lib"), "-lc10", "-lc10_hip", "-ltorch_cpu",
           "-ltorch_hip", "-ltorch", "-ltorch_python", "-Wl,-rpath,$ORIGIN"]
    _run(cmd, verbose)
    return TORCH_MODULE


def build_hostcheck(verbose: bool = False) -> str:
    os.makedirs(LIBDIR, exist_ok=True)
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Wno-unknown-pragmas", "-I", CSRC,
           os.path.join(CSRC, "ap_hostcheck.cpp"), "-o", HOSTCHECK_LIB]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    return HOSTCHECK_LIB


def build_all(verbose: bool = False) -> None:
    build_hip(verbose)
    build_torch(verbose)
    build_hostcheck(verbose)


if __name__ == "__main__":
    build_all(verbose=True)
    print("built:", HIP_LIB, TORCH_MODULE, HOSTCHECK_LIB)
