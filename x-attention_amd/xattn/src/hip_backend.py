"""Bindings of the native libraries: libxattn_hip.so (the kernels behind the C
ABI declared in include/xattn_hip.h, through ctypes) and xattn_host.so (the same
C ABI called straight from torch tensors, for the calls whose host time counts).

Both are built ahead of time by ``x-attention_amd/csrc/build.py``; if one is
missing, :func:`lib` / :func:`host` fail loudly - there is no fallback path.
"""
import ctypes
import importlib.machinery
import importlib.util
import os

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.normpath(os.path.join(_HERE, "..", "..", "csrc", "libxattn_hip.so"))

HOST_PATH = os.path.join(os.path.dirname(LIB_PATH), "xattn_host.so")

c_i32, c_i64, c_f32, c_vp, c_sz = ctypes.c_int, ctypes.c_int64, ctypes.c_float, ctypes.c_void_p, ctypes.c_size_t

_SIGNATURES = {
    "xattn_abi_version": (c_i32, []),
    "xattn_error_string": (ctypes.c_char_p, [c_i32]),
    "xattn_estimate_workspace_bytes": (c_sz, [c_i32] * 7),
    "xattn_estimate_block_sums": (
        c_i32,
        [c_vp, c_vp, c_vp, c_vp, c_sz, c_vp] + [c_i32] * 5 + [c_i64] * 4 + [c_i32] * 7
        + [c_f32, ctypes.POINTER(c_i32), c_i32, c_i32, c_i32, c_i32, c_i32, c_i32, c_vp],
    ),
    "xattn_estimate_select": (
        c_i32,
        [c_vp, c_vp, c_vp, c_vp, c_sz] + [c_i32] * 5 + [c_i64] * 4 + [c_i32] * 7
        + [c_f32, ctypes.POINTER(c_i32), c_i32, c_i32, c_i32, c_i32, c_i32]
        + [c_vp] * 4 + [c_i64, c_i32, c_i32, c_i32, c_vp],
    ),
    "xattn_select_blocks": (
        c_i32,
        [c_vp] * 5 + [c_i64] + [c_i32] * 15 + [c_vp],
    ),
    "xattn_calibration_copy": (c_i32, [c_vp, c_vp, c_sz, c_vp]),
    "xattn_mfma_rate_probe": (c_i32, [c_vp, c_i32, c_i32, c_vp, ctypes.POINTER(ctypes.c_double), c_vp]),
    "xattn_softmax_block_sums": (c_i32, [c_vp, c_vp] + [c_i32] * 3 + [c_i64] * 2 + [c_i32] * 3 + [c_f32, c_i32, c_vp]),
    "xattn_block_mass": (c_i32, [c_vp] * 3 + [c_i32] * 5 + [c_i64] * 4 + [c_i32, c_f32, c_vp]),
    "xattn_threshold_rows": (c_i32, [c_vp] * 3 + [c_i32] * 3 + [c_i64] * 2 + [c_f32, c_vp]),
    "xattn_prefill_workspace_bytes": (c_sz, [c_i32] * 5),
    "xattn_prefill_least_workspace_bytes": (c_sz, [c_i32] * 5),
    "xattn_prefill_fwd": (
        c_i32,
        [c_vp] * 5 + [c_sz] + [c_i32] * 5 + [c_i64] * 8 + [c_i32] * 4 + [c_f32, c_i32]
        + [ctypes.POINTER(ctypes.c_double), c_i32, c_vp, c_i32, c_i32, c_f32, c_vp],
    ),
    "xattn_estimate_fwd": (
        c_i32,
        [c_vp] * 5 + [c_sz] + [c_i32] * 5 + [c_i64] * 4 + [c_i32] * 4 + [c_f32, c_i32]
        + [ctypes.POINTER(ctypes.c_double), c_i32, c_vp, c_i32, c_i32, c_vp],
    ),
    "xattn_decode_workspace_bytes": (c_sz, [c_i32] * 3),
    "xattn_decode_fwd": (
        c_i32,
        [c_vp] * 5 + [c_sz] + [c_i32] * 4 + [c_i64] * 6 + [c_f32, c_vp],
    ),
    "xattn_decode_fwd_static": (
        c_i32,
        [c_vp] * 4 + [c_i32] * 4 + [c_i64] * 6 + [c_f32, c_vp],
    ),
    "xattn_qkv_rope_gemv": (
        c_i32,
        [c_vp, c_i32] + [c_vp, c_i64, c_vp] * 3 + [c_vp] * 5 + [c_i32] * 3 + [c_vp],
    ),
    "xattn_gemv": (c_i32, [c_vp, c_i32, c_vp, c_i64, c_vp, c_vp, c_i32, c_vp]),
    "xattn_proj_gemm_fits": (c_i32, [c_i32] * 4),
    "xattn_qkv_rope_gemm": (
        c_i32,
        [c_vp, c_i32, c_i32] + [c_vp, c_i64, c_vp] * 3 + [c_vp] * 2 + [c_i64] * 2 + [c_vp] * 3 + [c_i32] * 3 + [c_vp],
    ),
    "xattn_gemm": (c_i32, [c_vp, c_i32, c_i32, c_vp, c_i64, c_vp, c_vp, c_i32, c_vp]),
    "xattn_rope": (c_i32, [c_vp] * 4 + [c_i64] * 2 + [c_i32] * 4 + [c_vp]),
    "xattn_block_sparse_workspace_bytes": (c_sz, [c_i32] * 5),
    "xattn_block_sparse_fwd_ws": (
        c_i32,
        [c_vp] * 5 + [c_sz] + [c_vp] * 2 + [c_i64] + [c_i32] * 7 + [c_i64] * 8 + [c_i32, c_i32, c_i32, c_f32, c_vp],
    ),
    "xattn_block_sparse_fwd": (
        c_i32,
        [c_vp] * 6 + [c_i64] + [c_i32] * 7 + [c_i64] * 8 + [c_i32, c_i32, c_i32, c_f32, c_vp],
    ),
}

_lib = None
_host = None


class XattnHipError(RuntimeError):
    pass


def lib():
    """The loaded library; raises if it has not been built."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise XattnHipError(
                f"{LIB_PATH} is missing: build it with `python x-attention_amd/csrc/build.py` "
                "(there is no non-HIP fallback)"
            )
        handle = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in _SIGNATURES.items():
            fn = getattr(handle, name)
            fn.restype, fn.argtypes = res, args
        _lib = handle
    return _lib


def host():
    """The native host module; raises if it has not been built."""
    global _host
    if _host is None:
        lib()
        if not os.path.exists(HOST_PATH):
            raise XattnHipError(f"{HOST_PATH} is missing: build it with `python x-attention_amd/csrc/build.py`")
        loader = importlib.machinery.ExtensionFileLoader("xattn_host", HOST_PATH)
        module = importlib.util.module_from_spec(importlib.util.spec_from_loader("xattn_host", loader))
        loader.exec_module(module)
        _host = module
    return _host


def exported_symbols():
    return list(_SIGNATURES)


def check(code, what):
    if code != 0:
        msg = lib().xattn_error_string(code).decode()
        raise XattnHipError(f"{what} failed: {msg} (code {code})")
