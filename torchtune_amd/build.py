"""Compile the HIP sources in ``torchtune_amd/csrc`` into ``torchtune_amd/lib/libtorchtune_amd.so`` for gfx950.

The library is a plain C-ABI shared object (see ``include/torchtune_amd.h``); it links against the HIP
runtime only, never against torch.  Next to it goes ``torchtune_amd_host.so``, the extension module that makes layer
calls into it without the interpreter (``csrc/host_binding.cpp``).  ``python -m torchtune_amd.build`` rebuilds both.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
LIB_DIR = PKG / "lib"
LIB_PATH = LIB_DIR / "libtorchtune_amd.so"
HOST_MODULE = "torchtune_amd_host"
HOST_PATH = LIB_DIR / f"{HOST_MODULE}.so"
SOURCES = ["capi.hip", "nf4_codec.hip", "fake_quant.hip", "int4_linear.hip", "nf4_gemm.hip", "nf4_gemm_rs.hip", "nf4_gemm_mid.hip", "nf4_gemm_dense.hip", "gemm_tn.hip", "gemm_mid.hip", "nf4_small_m.hip", "lora_skinny.hip", "lora_group.hip", "qlora_linear.hip", "nf4_merge.hip", "neighbours.hip"]

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-fast-math",
    "-ffp-contract=off",  # quantisation results must not depend on fma contraction
    "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-fno-gpu-flush-denormals-to-zero",
    # packed fp32 VALU ops are kept out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
]


def hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found: the HIP toolchain (ROCm) is required to build torchtune_amd")
    return exe


def _compile(src: str, obj_dir: Path) -> Path:
    obj = obj_dir / (Path(src).stem + ".o")
    cmd = [hipcc(), *HIPCC_FLAGS, "-c", str(CSRC / src), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{proc.stdout}\n{proc.stderr}")
    return obj


def _compile_host(obj_dir: Path) -> Path:
    """The torch side of the C ABI (``csrc/host_binding.cpp``): host code only, compiled against torch's headers."""
    import torch
    from torch.utils.cpp_extension import include_paths

    obj = obj_dir / "host_binding.o"
    cmd = [
        shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function", "-D__HIP_PLATFORM_AMD__=1",
        "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f"-DTORCH_EXTENSION_NAME={HOST_MODULE}",
        *[f"-isystem{p}" for p in include_paths()], "-isystem/opt/rocm/include", f"-isystem{sysconfig.get_paths()['include']}",
        "-c", str(CSRC / "host_binding.cpp"), "-o", str(obj),
    ]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"g++ failed on host_binding.cpp:\n{proc.stdout}\n{proc.stderr}")
    return obj


def _link_host(obj: Path) -> None:
    import torch

    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    tmp = HOST_PATH.with_suffix(".so.tmp")
    cmd = [shutil.which("g++") or "g++", "-shared", "-o", str(tmp), str(obj), f"-L{LIB_DIR}", "-ltorchtune_amd", f"-L{torch_lib}", "-lc10",
           "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python", "-Wl,-rpath,$ORIGIN"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link of {HOST_PATH.name} failed:\n{proc.stdout}\n{proc.stderr}")
    os.replace(tmp, HOST_PATH)


def build(verbose: bool = False) -> Path:
    """Compile every source and link the shared library and the host extension. Always recompiles."""
    obj_dir = PKG / "build"
    obj_dir.mkdir(exist_ok=True)
    LIB_DIR.mkdir(exist_ok=True)
    with ThreadPoolExecutor(max_workers=min(len(SOURCES) + 1, 8)) as pool:
        host = pool.submit(_compile_host, obj_dir)
        objs = list(pool.map(lambda s: _compile(s, obj_dir), SOURCES))
        host_obj = host.result()
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed:\n{proc.stdout}\n{proc.stderr}")
    os.replace(tmp, LIB_PATH)
    _link_host(host_obj)
    if verbose:
        print(f"built {LIB_PATH} and {HOST_PATH.name}")
    return LIB_PATH


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
