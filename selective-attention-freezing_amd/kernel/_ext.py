"""ctypes binding of libsafattn.so (C-ABI declared in include/saf_attn.h).

The library is built in-tree by ``build_ext.build()`` and loaded from this
directory.  There is no fallback: if the library is missing, every entry point
that needs it raises ``RuntimeError`` naming the build step.
"""
import ctypes
import os
import struct

import numpy as np
import torch

LIB_NAME = "libsafattn.so"
LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), LIB_NAME)

SAF_OK, SAF_EINVAL, SAF_EUNSUPPORTED, SAF_EALIGN, SAF_ELAUNCH, SAF_EWORKSPACE = 0, -1, -2, -3, -4, -5
SAF_F32, SAF_F16, SAF_BF16, SAF_I32 = 0, 1, 2, 3
SAF_MAX_HEADS = 128

_DTYPE_CODE = {torch.float32: SAF_F32, torch.float16: SAF_F16,
               torch.bfloat16: SAF_BF16, torch.int32: SAF_I32}

# Exported symbols, in header order (checked by the CPU test suite).
EXPORTS = ("saf_mixed_attn_fwd", "saf_mixed_attn_side_kernels", "saf_mixed_attn_fwd_noalloc", "saf_flash_fwd",
           "saf_frozen_dense_pv_fwd", "saf_frozen_decomp_fwd", "saf_frozen_scan_fwd", "saf_mixed_attn_bwd",
           "saf_mixed_attn_bwd_workspace_bytes", "saf_decomp_param_bwd", "saf_decomp_param_bwd_workspace_bytes",
           "saf_frozen_pv_fwd", "saf_frozen_pv_bwd",
           "saf_rope_qk_inplace", "saf_qk_rmsnorm_rope_inplace", "saf_add_layernorm",
           "saf_add_rmsnorm", "saf_linear_gelu", "saf_gelu_inplace", "saf_linear_swiglu", "saf_linear_rope", "saf_decomposed_logz",
           "saf_decomposed_logz_bwd", "saf_workspace_bytes", "saf_mixed_attn_workspace_bytes", "saf_workspace_error",
           "saf_time_next_kernel", "saf_last_error", "saf_version")


class SafTensor(ctypes.Structure):
    _fields_ = [("data", ctypes.c_void_p), ("dtype", ctypes.c_int32),
                ("ndim", ctypes.c_int32), ("size", ctypes.c_int64 * 4),
                ("stride", ctypes.c_int64 * 4)]


class SafMixedAttnArgs(ctypes.Structure):
    _fields_ = [("q", SafTensor), ("k", SafTensor), ("v", SafTensor),
                ("out", SafTensor), ("lse", SafTensor), ("patt", SafTensor),
                ("alpha", SafTensor), ("rho", SafTensor), ("z", SafTensor),
                ("n_heads", ctypes.c_int32),
                ("frozen", ctypes.POINTER(ctypes.c_int32)),
                ("hidx", ctypes.POINTER(ctypes.c_int32)),
                ("pidx", ctypes.POINTER(ctypes.c_int32)),
                ("kvidx", ctypes.POINTER(ctypes.c_int32)),
                ("closed_kind", ctypes.POINTER(ctypes.c_int32)),
                ("closed_param", ctypes.POINTER(ctypes.c_float)),
                ("sm_scale", ctypes.c_float),
                ("workspace", ctypes.c_void_p),
                ("workspace_bytes", ctypes.c_int64),
                ("flash_qtiles", ctypes.c_int32),
                ("scan_spin_limit", ctypes.c_int32),
                ("decomp_unsplit", ctypes.c_int32)]


_lib = None


def available():
    """True if libsafattn.so has been built next to this module."""
    return os.path.exists(LIB_PATH)


def lib():
    """The loaded library (loaded once per process)."""
    global _lib
    if _lib is None:
        if not available():
            raise RuntimeError(
                f"{LIB_NAME} is not built ({LIB_PATH} missing): run "
                "__graft_entry__.build() (or build_ext.build()) first; the SAF "
                "operators have no non-HIP fallback")
        L = ctypes.CDLL(LIB_PATH)
        P = ctypes.POINTER
        for name in ("saf_mixed_attn_fwd", "saf_mixed_attn_fwd_noalloc", "saf_flash_fwd", "saf_frozen_dense_pv_fwd",
                     "saf_frozen_decomp_fwd", "saf_frozen_scan_fwd"):
            fn = getattr(L, name)
            fn.argtypes = [P(SafMixedAttnArgs), ctypes.c_void_p]
            fn.restype = ctypes.c_int
        L.saf_mixed_attn_side_kernels.argtypes = [P(SafMixedAttnArgs)]
        L.saf_mixed_attn_side_kernels.restype = ctypes.c_int
        L.saf_mixed_attn_bwd.argtypes = [P(SafMixedAttnArgs)] + [P(SafTensor)] * 4 + [ctypes.c_void_p]
        L.saf_mixed_attn_bwd.restype = ctypes.c_int
        L.saf_mixed_attn_bwd_workspace_bytes.argtypes = [P(SafMixedAttnArgs)]
        L.saf_mixed_attn_bwd_workspace_bytes.restype = ctypes.c_int64
        L.saf_decomp_param_bwd.argtypes = [P(SafMixedAttnArgs)] + [P(SafTensor)] * 3 + [ctypes.c_void_p]
        L.saf_decomp_param_bwd.restype = ctypes.c_int
        L.saf_decomp_param_bwd_workspace_bytes.argtypes = [P(SafMixedAttnArgs)]
        L.saf_decomp_param_bwd_workspace_bytes.restype = ctypes.c_int64
        L.saf_frozen_pv_fwd.argtypes = [P(SafTensor), P(SafTensor), P(ctypes.c_int32),
                                        ctypes.c_int32, ctypes.c_int32, P(SafTensor),
                                        ctypes.c_void_p]
        L.saf_frozen_pv_fwd.restype = ctypes.c_int
        L.saf_frozen_pv_bwd.argtypes = L.saf_frozen_pv_fwd.argtypes
        L.saf_frozen_pv_bwd.restype = ctypes.c_int
        L.saf_rope_qk_inplace.argtypes = [P(SafTensor)] * 4 + [ctypes.c_void_p]
        L.saf_rope_qk_inplace.restype = ctypes.c_int
        L.saf_qk_rmsnorm_rope_inplace.argtypes = [P(SafTensor)] * 4 + [ctypes.c_float] + \
            [P(SafTensor)] * 2 + [ctypes.c_void_p]
        L.saf_qk_rmsnorm_rope_inplace.restype = ctypes.c_int
        L.saf_add_layernorm.argtypes = [P(SafTensor)] * 4 + [ctypes.c_float, P(SafTensor), ctypes.c_void_p]
        L.saf_add_layernorm.restype = ctypes.c_int
        L.saf_add_rmsnorm.argtypes = [P(SafTensor)] * 3 + [ctypes.c_float, P(SafTensor), ctypes.c_void_p]
        L.saf_add_rmsnorm.restype = ctypes.c_int
        L.saf_linear_gelu.argtypes = [P(SafTensor)] * 3 + [ctypes.c_void_p]
        L.saf_linear_gelu.restype = ctypes.c_int
        L.saf_gelu_inplace.argtypes = [P(SafTensor), ctypes.c_void_p]
        L.saf_gelu_inplace.restype = ctypes.c_int
        L.saf_linear_swiglu.argtypes = [P(SafTensor)] * 3 + [ctypes.c_void_p]
        L.saf_linear_swiglu.restype = ctypes.c_int
        L.saf_linear_rope.argtypes = [P(SafTensor)] * 3 + [ctypes.c_int32] * 3 + [P(SafTensor)] * 2 + [ctypes.c_void_p]
        L.saf_linear_rope.restype = ctypes.c_int
        L.saf_decomposed_logz.argtypes = [P(SafTensor)] * 3 + [ctypes.c_void_p]
        L.saf_decomposed_logz.restype = ctypes.c_int
        L.saf_decomposed_logz_bwd.argtypes = [P(SafTensor)] * 6 + [ctypes.c_void_p]
        L.saf_decomposed_logz_bwd.restype = ctypes.c_int
        L.saf_workspace_bytes.argtypes = [ctypes.c_int32] * 4
        L.saf_workspace_bytes.restype = ctypes.c_int64
        L.saf_mixed_attn_workspace_bytes.argtypes = [P(SafMixedAttnArgs)]
        L.saf_mixed_attn_workspace_bytes.restype = ctypes.c_int64
        L.saf_workspace_error.argtypes = [ctypes.c_void_p, ctypes.c_void_p, P(ctypes.c_int32)]
        L.saf_workspace_error.restype = ctypes.c_int
        L.saf_time_next_kernel.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
        L.saf_time_next_kernel.restype = ctypes.c_int
        L.saf_last_error.argtypes = []
        L.saf_last_error.restype = ctypes.c_char_p
        L.saf_version.argtypes = []
        L.saf_version.restype = ctypes.c_char_p
        _lib = L
    return _lib


# saf_tensor_t packed in one go: a descriptor filled field by field through
# ctypes cost 2.3 us a tensor, packed 1.1 us, packed into its place in the
# argument block 0.9 us (a call has four to nine of them)
_DESC = struct.Struct("@Pii8q")
_PAD = tuple((0,) * (4 - n) for n in range(5))


def _desc_values(t):
    shape = t.shape
    n = len(shape)
    if n > 4:
        raise ValueError("SAF tensors have at most 4 dimensions")
    code = _DTYPE_CODE.get(t.dtype)
    if code is None:
        raise NotImplementedError(f"unsupported dtype {t.dtype}")
    if n == 4:
        return (t.data_ptr(), code, 4, *shape, *t.stride())
    return (t.data_ptr(), code, n, *shape, *_PAD[n], *t.stride(), *_PAD[n])


def tensor_desc(t):
    """saf_tensor_t for a torch tensor (None -> an absent descriptor)."""
    if t is None:
        return SafTensor()
    return SafTensor.from_buffer_copy(_DESC.pack(*_desc_values(t)))


def rows_desc(t):
    """tensor_desc(t.view(-1, C)) of an activation (..., C)."""
    if not t.is_contiguous() or t.dtype not in _DTYPE_CODE or t.numel() == 0:
        return tensor_desc(t.view(-1, t.size(-1)))
    C = t.shape[-1]
    return SafTensor.from_buffer_copy(_DESC.pack(t.data_ptr(), _DTYPE_CODE[t.dtype], 2, t.numel() // C, C, 0, 0,
                                                 C, 1, 0, 0))


def set_desc(args, offset, t):
    """tensor_desc(t) written at a byte offset of an argument block."""
    _DESC.pack_into(args, offset, *_desc_values(t))


# saf_mixed_attn_args: offsets of the tensor descriptors, and the fields from
# n_heads to closed_param, from sm_scale on
ARG_OFFSET = {n: getattr(SafMixedAttnArgs, n).offset
              for n in ("q", "k", "v", "out", "lse", "patt", "alpha", "rho", "z")}
_TABLES = struct.Struct("@i6P")
_WORKSPACE = struct.Struct("@Pq")


def set_tables(args, n_heads, *tables):
    """n_heads and the six routing tables (ctypes arrays or None), which the
    caller keeps alive as long as the block is used."""
    _TABLES.pack_into(args, SafMixedAttnArgs.n_heads.offset, n_heads,
                      *[0 if t is None else ctypes.addressof(t) for t in tables])


def set_workspace(args, ptr, nbytes):
    _WORKSPACE.pack_into(args, SafMixedAttnArgs.workspace.offset, ptr, nbytes)


def check(rc):
    """Raise the Python exception matching a C-ABI status."""
    if rc == SAF_OK:
        return
    msg = lib().saf_last_error().decode(errors="replace")
    if rc == SAF_EUNSUPPORTED:
        raise NotImplementedError(msg)
    if rc in (SAF_EINVAL, SAF_EALIGN, SAF_EWORKSPACE):
        raise ValueError(msg)
    raise RuntimeError(msg)


def _host_array(values, ctype, dtype):
    if values is None:
        return None
    arr = np.ascontiguousarray(values, dtype=dtype)
    return (ctype * arr.size).from_buffer_copy(arr) if arr.size else (ctype * 0)()


def host_i32(values):
    """ctypes int32 array from a host sequence / numpy array (None passes)."""
    return _host_array(values, ctypes.c_int32, np.int32)


def host_f32(values):
    return _host_array(values, ctypes.c_float, np.float32)


def current_stream_ptr(device):
    """Raw handle of the device's current stream."""
    index = device.index
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device() if index is None else index)
