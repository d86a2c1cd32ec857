"""Builds libbhi_hip.so for gfx950 next to the package (python -m bf16_huffman_infer_amd.csrc.build)."""
import os
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.dirname(HERE)
SOURCES = ["bhi_api.hip", "bhi_huffman.hip", "bhi_ans.hip", "bhi_nibble.hip", "bhi_reference.hip", "bhi_attention.hip",
           "bhi_convert.hip"]
LIB = os.path.join(PKG, "libbhi_hip.so")
TORCH_SOURCE = "bhi_torch.cpp"                       # host code alone: compiled against torch and Python, links no kernel
TORCH_LIB = os.path.join(PKG, "_bhi_torch.so")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # the first five dwords of every kernel's arguments arrive in registers (the fused GEMV
    # picks its group member from them before its first memory access)
    "-mllvm", "-amdgpu-kernarg-preload-count=5",
    "-Wall", "-Wno-unused-variable",
]


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    out = "\n".join(l for l in (proc.stdout + proc.stderr).splitlines() if "packed-fp32-ops" not in l)
    if verbose and out.strip():
        print(out)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed ({proc.returncode}):\n{out}")


def build(verbose: bool = True, defines=(), lib: str = LIB) -> str:
    """Compiles every source to an object of its own (in parallel) and links them."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    with tempfile.TemporaryDirectory(prefix="bhi_build_") as tmp:
        objs = [os.path.join(tmp, s.replace(".hip", ".o")) for s in SOURCES]
        cmds = [[hipcc, *FLAGS, *[f"-D{d}" for d in defines], "-c", os.path.join(HERE, s), "-o", o]
                for s, o in zip(SOURCES, objs)]
        with ThreadPoolExecutor(max_workers=min(len(cmds), os.cpu_count() or 1)) as pool:
            list(pool.map(lambda c: _run(c, verbose), cmds))
        _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", lib], verbose)
    return lib


def build_torch(verbose: bool = True, lib: str = TORCH_LIB) -> str:
    import sysconfig

    import torch
    root = os.path.dirname(torch.__file__)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    _run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
          "-isystem", os.path.join(root, "include"), "-isystem", os.path.join(root, "include", "torch", "csrc", "api", "include"),
          "-isystem", os.path.join(rocm, "include"), "-isystem", sysconfig.get_paths()["include"],
          os.path.join(HERE, TORCH_SOURCE), "-o", lib, "-L" + os.path.join(root, "lib"),
          "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch_python"], verbose)
    return lib


if __name__ == "__main__":
    build()
    build_torch()
    sys.exit(0)
