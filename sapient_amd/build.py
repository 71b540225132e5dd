"""Build the gfx950 shared library ``sapient_amd/libsapient_hip.so``.

Each ``csrc/*.hip`` / ``csrc/*.cpp`` kernel translation unit and the C++
host layer (``host/*.cpp``) is compiled by hipcc (in parallel) into
``sapient_amd/_build/`` and linked into one shared library that exports the C
ABI declared in ``include/sapient_hip.h`` and the C++ API of
``include/sapient_hip_backend.hpp``. The native half of :mod:`sapient_amd.ops`
(``binding/torch_ops.cpp``, against the headers of Python and of the installed
torch) is compiled into ``sapient_amd/_torch_ops.so``, which links that library;
where torch or Python's headers are missing it is left out, with a note: the
library needs hipcc alone.

Usage: ``python -m sapient_amd.build`` (or ``__graft_entry__.build()``).
"""
from __future__ import annotations

import concurrent.futures as cf
import importlib.util
import os
import shutil
import subprocess
import sys
import sysconfig
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
BUILD = PKG / "_build"
LIB = PKG / "libsapient_hip.so"
BINDING = PKG / "_torch_ops.so"

ARCH = "gfx950"

# Numerics flags are part of the parity contract:
#  -ffp-contract=off      no a*b+c fusion: products and sums round as in the reference
#  correctly-rounded f32 divide/sqrt, f32 denormals kept (both HIP defaults, stated)
#  -packed-fp32-ops off   no v_pk_{add,mul,fma}_f32 generation
#  -fma-mix/-mad-mix off  no v_fma_mix*/v_mad_mix*: the backend folds f32 products
#                         into these f16-result ops, which round differently from
#                         "round to f32, then to f16" and give +0 for -0 products
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-fno-gpu-flush-denormals-to-zero",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Xclang", "-target-feature", "-Xclang", "-fma-mix-insts",
    "-Xclang", "-target-feature", "-Xclang", "-mad-mix-insts",
    "-Wall",
    "-Wno-unused-function",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found (expected /opt/rocm/bin/hipcc)")


def sources() -> list[Path]:
    return sorted(list(CSRC.glob("*.hip")) + list(CSRC.glob("*.cpp")) + list((PKG / "host").glob("*.cpp")))


def _compile(src: Path) -> Path:
    obj = BUILD / (src.stem + ".o")
    cmd = [hipcc(), *HIPCC_FLAGS, f"-I{ROOT / 'include'}", f"-I{CSRC}", "-c", str(src), "-o", str(obj)]
    if src.suffix == ".cpp":
        cmd[1:1] = ["-x", "hip"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{res.stderr}")
    return obj


def _build_binding() -> str:
    """The torch binding: host code only, in torch's own C++ ABI, found beside the library at run time.
    Returns why it was left out, or "". It records the torch and the ABI it was built for (ops.py checks both)."""
    include = Path(sysconfig.get_paths()["include"])
    missing = ("torch" if importlib.util.find_spec("torch") is None else
               "Python.h" if not (include / "Python.h").exists() else "")
    if missing:
        BINDING.unlink(missing_ok=True)  # one from an earlier build would be for another library
        return f"{missing} not found"
    import torch
    t = Path(torch.__file__).parent
    tmp = BINDING.with_suffix(".so.tmp")
    cmd = [shutil.which("g++") or hipcc(), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
           f'-DSPH_TORCH_VERSION="{torch.__version__}"', f"-I{ROOT / 'include'}",
           "-isystem", str(t / "include"), "-isystem", str(t / "include" / "torch" / "csrc" / "api" / "include"),
           "-isystem", "/opt/rocm/include", "-isystem", str(include),
           str(PKG / "binding" / "torch_ops.cpp"), "-o", str(tmp), f"-L{PKG}", f"-l:{LIB.name}", f"-L{t / 'lib'}",
           "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip", "-Wl,-rpath,$ORIGIN"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed for torch_ops.cpp:\n{res.stderr}")
    os.replace(tmp, BINDING)
    return ""


def build(verbose: bool = True) -> Path:
    """Compile every translation unit for gfx950 and link the shared library."""
    BUILD.mkdir(exist_ok=True)
    srcs = sources()
    workers = max(1, min(len(srcs), os.cpu_count() or 1, 8))
    with cf.ThreadPoolExecutor(workers) as ex:
        objs = list(ex.map(_compile, srcs))
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp),
           "-Wl,-rpath,/opt/rocm/lib"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    os.replace(tmp, LIB)
    left_out = _build_binding()
    if verbose:
        print(f"built {LIB.relative_to(ROOT)} from {len(srcs)} sources")
        if left_out:
            print(f"left out {BINDING.relative_to(ROOT)}, the calls on torch tensors: {left_out}")
    return LIB


if __name__ == "__main__":
    build()
    sys.exit(0)
