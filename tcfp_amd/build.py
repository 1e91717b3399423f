"""Build ``libtcfp_hip.so`` (hand-written HIP for gfx950) in-tree.

    python -m tcfp_amd.build

Each ``csrc/*.hip`` file is compiled by ``hipcc --offload-arch=gfx950`` to
an object under ``tcfp_amd/_build/`` and the objects are linked into
``tcfp_amd/libtcfp_hip.so``.  The library has no libtorch dependency: the
Python side binds it through ctypes, and through ``tcfp_amd/_tcfp_host.so``
(``csrc/host.cpp``, host C++ against torch's headers and the library), the
native host path of the ops that every layer pass makes.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
BUILD = PKG / "_build"
LIB = PKG / "libtcfp_hip.so"
HOST = PKG / "_tcfp_host.so"
INCLUDE = PKG.parent / "include"

ARCH = "gfx950"

COMMON_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    f"-I{INCLUDE}",
    # packed fp32 VALU ops are kept out of the generated code: some of their
    # forms have given wrong results on MI355X without any error; hipcc's
    # host pass warns it does not know the feature, which is harmless.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]

# Per-file extra flags.  The quantisation kernels and the GEMM epilogues
# that evaluate GELU must match torch's separately rounded elementwise ops
# bit for bit (and each other: the erf / exp they inline are compiled with
# these flags too): no contraction to FMA.
EXTRA = {
    "quant.hip": ["-ffp-contract=off"],
    "gemm.hip": ["-ffp-contract=off"],
}


def hipcc() -> str:
    cand = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(cand).exists():
        raise RuntimeError("hipcc not found: the HIP toolchain (ROCm) is required to build")
    return cand


def host_commands(obj: Path, out: Path) -> tuple[list[str], list[str]]:
    """Compile and link commands of the native host module (no GPU code)."""
    import torch
    from torch.utils import cpp_extension as ext

    cxx = shutil.which("g++") or "g++"
    inc = [*ext.include_paths(), sysconfig.get_paths()["include"], "/opt/rocm/include"]
    compile_ = [
        cxx, "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
        f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
        *(f"-I{i}" for i in inc), "-c", str(CSRC / "host.cpp"), "-o", str(obj),
    ]
    link = [
        cxx, "-shared", str(obj), "-o", str(out), *(f"-L{p}" for p in ext.library_paths()),
        "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip", f"-L{PKG}",
        "-ltcfp_hip", "-Wl,-rpath,$ORIGIN",
    ]
    return compile_, link


def build(verbose: bool = True) -> Path:
    BUILD.mkdir(exist_ok=True)
    cc = hipcc()
    sources = sorted(CSRC.glob("*.hip"))
    procs = []
    objs = []
    for src in sources:
        obj = BUILD / (src.stem + ".o")
        objs.append(obj)
        cmd = [cc, *COMMON_FLAGS, *EXTRA.get(src.name, []), "-c", str(src), "-o", str(obj)]
        if verbose:
            print("[tcfp_amd.build]", " ".join(cmd), flush=True)
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)))
    host_tmp = HOST.with_suffix(".so.tmp")
    host_cc, host_link = host_commands(BUILD / "host.o", host_tmp)
    if verbose:
        print("[tcfp_amd.build]", " ".join(host_cc), flush=True)
    procs.append((CSRC / "host.cpp",
                  subprocess.Popen(host_cc, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)))
    failed = []
    for src, p in procs:
        out, _ = p.communicate()
        text = out.decode(errors="replace")
        text = "\n".join(l for l in text.splitlines() if "packed-fp32-ops" not in l)
        if p.returncode != 0:
            failed.append((src, text))
        elif text.strip() and verbose:
            print(text, flush=True)
    if failed:
        msg = "\n".join(f"--- {s.name} ---\n{t}" for s, t in failed)
        raise RuntimeError(f"HIP build failed:\n{msg}")
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [cc, f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)]
    if verbose:
        print("[tcfp_amd.build]", " ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    os.replace(tmp, LIB)
    if verbose:
        print("[tcfp_amd.build]", " ".join(host_link), flush=True)
    subprocess.run(host_link, check=True)
    os.replace(host_tmp, HOST)
    return LIB


if __name__ == "__main__":
    build(verbose="-q" not in sys.argv)
