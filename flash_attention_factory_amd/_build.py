"""Compiles the HIP library for gfx950 in-tree (hipcc cross-compiles without a GPU)."""
from __future__ import annotations

import os
import subprocess

_PKG = os.path.dirname(os.path.abspath(__file__))
SOURCE = os.path.join(_PKG, "csrc", "fa_paged_attention.hip")
LIBRARY = os.path.join(_PKG, "libfa_paged_attention.so")

TORCH_OPS_SOURCE = os.path.join(_PKG, "csrc", "torch_ops.cpp")
TORCH_OPS_LIBRARY = os.path.join(_PKG, "libfa_torch_ops.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
    # packed-fp32 instructions are kept out of the generated code on purpose
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
]


def build(verbose: bool = False, extra_flags=(), output: str = LIBRARY) -> str:
    """The product library, or with extra_flags and another output a debug build beside it
    (-DFA_TIMELINE: in-kernel timeline; -DFA_COST_PROBE=1|2: the segment kernels without their stores
    of partials), which FA_PAGED_ATTENTION_LIBRARY selects at run time."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    cmd = [hipcc, *HIPCC_FLAGS, *extra_flags, SOURCE, "-o", output]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed ({res.returncode}):\n{res.stdout}\n{res.stderr}")
    return output


def build_torch_ops(verbose: bool = False, output: str = TORCH_OPS_LIBRARY) -> str:
    """The native operators of torch.ops.fa_amd (host code only)."""
    import torch
    root = os.path.dirname(torch.__file__)
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-fvisibility=hidden",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           "-isystem", os.path.join(root, "include"), "-isystem", os.path.join(root, "include", "torch", "csrc", "api", "include"),
           "-isystem", "/opt/rocm/include", TORCH_OPS_SOURCE, "-o", output, "-L" + os.path.join(root, "lib"),
           "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip"]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed ({res.returncode}):\n{res.stdout}\n{res.stderr}")
    return output


if __name__ == "__main__":
    import argparse
    ap = argparse.ArgumentParser(description=__doc__)
    ap.add_argument("--output", default=LIBRARY)
    args, flags = ap.parse_known_args()  # everything else goes to hipcc (-DFA_TIMELINE ...)
    print(build(verbose=True, extra_flags=flags, output=os.path.abspath(args.output)))
    if not flags and os.path.abspath(args.output) == LIBRARY:
        print(build_torch_ops(verbose=True))
