"""Builds libxattn_hip.so (gfx950 kernels behind the C ABI) and xattn_host.so
(the Python package's native host path) next to their sources.

    python x-attention_amd/csrc/build.py

The libraries are built in-tree so that they travel with the source tree; nothing
is compiled at import time.
"""
import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
SOURCES = ["capi.hip", "block_sparse_attn.hip", "estimate.hip", "select_blocks.hip", "decode_attn.hip", "profile_threshold.hip", "softmax_block_sum.hip",
           "prefill.hip", "layer_proj.hip", "proj_gemm.hip"]
LIB = os.path.join(HERE, "libxattn_hip.so")
HOST_SOURCE = os.path.join(HERE, "host_torch.cpp")
HOST_LIB = os.path.join(HERE, "xattn_host.so")
FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Wno-unused-result",
    "-Wno-inline-asm",   # the tile copies name M0 (their LDS destination) in an asm clobber list
    "-I" + os.path.join(ROOT, "include"),
    "-I" + HERE,
    # packed fp32 VALU forms are kept out of every kernel
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def _run(cmd):
    proc = subprocess.run(cmd, cwd=HERE, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in proc.stdout.splitlines() if "packed-fp32-ops" not in l)
    if proc.returncode != 0:
        raise RuntimeError("command failed: " + " ".join(cmd) + "\n" + out)
    return out


def build_host():
    """The CPython module over torch's C++ tensors; finds libxattn_hip.so beside itself."""
    import torch

    tdir = os.path.dirname(torch.__file__)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    return _run([
        os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
        f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
        "-I" + os.path.join(ROOT, "include"), "-I" + HERE,
        "-isystem", os.path.join(tdir, "include"), "-isystem", os.path.join(tdir, "include", "torch", "csrc", "api", "include"),
        "-isystem", os.path.join(rocm, "include"), "-isystem", sysconfig.get_paths()["include"],
        HOST_SOURCE, "-o", HOST_LIB, "-L" + HERE, "-lxattn_hip", "-L" + os.path.join(tdir, "lib"),
        "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip", "-Wl,-rpath,$ORIGIN",
    ])


def build(verbose=True):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    extra = os.environ.get("XATTN_HIPCC_EXTRA", "").split()
    srcs = [s for s in SOURCES if os.path.exists(os.path.join(HERE, s))]
    objs = [os.path.join(HERE, s.replace(".hip", ".o")) for s in srcs]

    def compile_one(pair):
        src, obj = pair
        return _run([hipcc] + FLAGS + extra + ["-c", src, "-o", obj])

    with ThreadPoolExecutor(max_workers=4) as ex:
        outs = list(ex.map(compile_one, zip(srcs, objs)))
    outs.append(_run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, "-Wl,-soname,libxattn_hip.so"] + objs))
    outs.append(build_host())
    if verbose:
        for o in outs:
            if o.strip():
                print(o)
        print("built", LIB, HOST_LIB)
    return LIB


if __name__ == "__main__":
    build()
    sys.exit(0)
