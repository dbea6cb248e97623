"""Builds libissm_hip.so (gfx950, hipcc) and _issm_host.so (the operators' host side on PyTorch tensors, g++) in-tree.
`python -m dest3d_amd.build`."""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libissm_hip.so")
HOST = os.path.join(HERE, "_issm_host.so")
SOURCES = ["issm_abi.hip", "issm_fwd.hip", "issm_fwd_tile.hip", "issm_bwd.hip", "issm_bwd_tile.hip", "issm_bwd_walk.hip", "issm_state_pass.hip", "rmsnorm_gated.hip", "param_gen.hip", "dwconv_silu.hip", "box_dist.hip", "box_dist_sorted.hip", "hilbert.hip", "pointnet2_ops.hip", "transpose_states.hip", "layer_params.hip", "linear.hip", "linear_tile.hip", "linear_dw.hip", "layer_out.hip"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffast-math", "-fno-finite-math-only",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument", "-Wno-unknown-attributes",
]


# Sources whose results are integers decided by floating-point comparisons, compiled without -ffast-math:
#  - hilbert.hip: a floating-point quotient picks the cell; IEEE division (no reciprocal-multiply rewriting) puts a
#    point exactly on a cell boundary into the same cell as on the host;
#  - pointnet2_ops.hip: squared distances pick indices (furthest point, ball membership, three nearest).  Under
#    -ffast-math the backend fuses multiply and add whatever `#pragma clang fp contract(off)` says, and a distance one
#    unit in the last place off decides a near-tie differently from a plain fp32 evaluation.
# and one that computes no more than a few exponentials, which are to be the accurate ones: layer_params.hip.
EXACT_ARITHMETIC = {"hilbert.hip", "pointnet2_ops.hip", "layer_params.hip", "linear.hip"}


def _compile(src: str) -> str:
    obj = os.path.join(CSRC, src.replace(".hip", ".o"))
    flags = [f for f in FLAGS if f not in ("-ffast-math", "-fno-finite-math-only")] if src in EXACT_ARITHMETIC else FLAGS
    cmd = [HIPCC, *flags, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _run(cmd, what: str) -> None:
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{what} failed:\n{r.stderr}")


def _compile_host() -> str:
    import torch
    t = os.path.dirname(torch.__file__)
    obj = os.path.join(CSRC, "host_ops.o")
    inc = [os.path.join(t, "include"), os.path.join(t, "include", "torch", "csrc", "api", "include"),
           sysconfig.get_path("include"), "/opt/rocm/include"]
    _run(["g++", "-O2", "-std=c++17", "-fPIC", *("-I" + i for i in inc), "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
          "-DTORCH_EXTENSION_NAME=_issm_host", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
          "-c", os.path.join(CSRC, "host_ops.cpp"), "-o", obj], "g++ host_ops.cpp")
    return obj


def _link_host(obj: str) -> None:
    import torch
    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    _run(["g++", "-shared", obj, "-o", HOST, "-L" + HERE, "-l:libissm_hip.so", "-L" + lib, "-ltorch", "-ltorch_cpu",
          "-ltorch_python", "-lc10", "-lc10_hip", "-Wl,-rpath,$ORIGIN"], "link of _issm_host.so")


def build(verbose: bool = True) -> str:
    """Compile every HIP source for gfx950 and the host side, link both shared libraries; returns the HIP library's path."""
    with ThreadPoolExecutor(max_workers=4) as ex:
        host = ex.submit(_compile_host)
        objs = list(ex.map(_compile, SOURCES))
        host_obj = host.result()
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", LIB]
    _run(cmd, "link")
    _link_host(host_obj)
    if verbose:
        print(f"built {LIB} and {HOST}")
    return LIB


if __name__ == "__main__":
    build()
