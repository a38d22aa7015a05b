"""ctypes binding of libfa2_fwd.so, the C ABI declared in include/fa2_fwd.h.

The library is built in-tree by triton-fa2-forward_amd/csrc/build.py and sits next to this
file. torch is imported first so that its HIP runtime (SONAME libamdhip64.so.7) is the one
already loaded when the library is opened: the library then launches on exactly the streams
torch hands out.
"""

import ctypes
import os
import sys

import torch  # noqa: F401  (must be loaded before the HIP library, see above)

LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libfa2_fwd.so")

# C-ABI symbols declared in include/fa2_fwd.h, with (restype, argtypes).
_i32, _i64p, _vp = ctypes.c_int32, ctypes.POINTER(ctypes.c_int64), ctypes.c_void_p
SIGNATURES = {
    "fa2_attn_fwd": (ctypes.c_int, [_vp, _vp, _vp, _vp, _i64p, _i64p, _i64p, _i64p,
                                    _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32,
                                    _i32, _i32, ctypes.c_float, _vp]),
    "fa2_attn_fwd_ex": (ctypes.c_int, [_vp, _vp, _vp, _vp, _i64p, _i64p, _i64p, _i64p,
                                       _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32,
                                       _i32, _i32, ctypes.c_float, _vp, _i32, _vp,
                                       ctypes.c_size_t, _vp]),
    "fa2_attn_fwd_noalloc": (ctypes.c_int, [_vp, _vp, _vp, _vp, _i64p, _i64p, _i64p, _i64p,
                                            _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32,
                                            _i32, _i32, ctypes.c_float, _vp, _i32, _vp]),
    "fa2_workspace_bytes": (ctypes.c_size_t, [_i32, _i32, _i32, _i32, _i32]),
    "fa2_workspace_bytes_for": (ctypes.c_size_t, [_i32, _i32, _i32, _i32, _i32, _i32, _i32,
                                                  _i32, _i32]),
    "fa2_num_splits": (_i32, [_i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _i32]),
    "fa2_launch_splits": (_i32, [_i32] * 11),
    "fa2_default_config": (ctypes.c_int, [_i32, ctypes.POINTER(_i32), ctypes.POINTER(_i32),
                                          ctypes.POINTER(_i32), ctypes.POINTER(_i32)]),
    "fa2_should_pack_gqa": (ctypes.c_int, [_i32, _i32, _i32]),
    "fa2_last_error": (ctypes.c_char_p, []),
    "fa2_version": (ctypes.c_char_p, []),
}

DTYPE_CODE = {torch.float16: 0, torch.bfloat16: 1}

_LIB = None


def lib():
    """The loaded library. Raises RuntimeError when it has not been built."""
    global _LIB
    if _LIB is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                f"{LIB_PATH} is missing; build the HIP library first: "
                "python triton-fa2-forward_amd/csrc/build.py")
        handle = ctypes.CDLL(LIB_PATH)
        for name, (restype, argtypes) in SIGNATURES.items():
            fn = getattr(handle, name)
            fn.restype = restype
            fn.argtypes = argtypes
        _LIB = handle
    return _LIB


def build_id():
    """The torch and the Python that the native call must have been built for: it reads tensors by
    their C++ layout, which another build of either can change without a missing symbol."""
    return "torch {} {} python {}.{}".format(torch.__version__, torch.version.git_version,
                                             *sys.version_info[:2])


def _load_fast_call():
    """The native common call of attention() (csrc/fa2_torch.cpp), built beside the library; None where
    it is missing or was built for another torch or Python: attention() then makes every call itself,
    through ctypes."""
    try:
        from . import _torch_call
    except ImportError:
        return None
    return _torch_call.call if getattr(_torch_call, "built_for", None) == build_id() else None


fast_call = _load_fast_call()


def last_error():
    return lib().fa2_last_error().decode(errors="replace")


_STRIDES = {}


def _strides(t):
    """The element strides as the C array the ABI takes. The stride of a size-1 dimension never
    enters an address; pass 0 so that only the strides the kernel actually steps by are checked
    against the 16-byte rule. The arrays are cached per (shape, strides): the library only reads
    them during the call, and building one costs more than the rest of a small call."""
    key = (t.shape, t.stride())
    arr = _STRIDES.get(key)
    if arr is None:
        if len(_STRIDES) >= 1024:
            _STRIDES.clear()
        arr = (ctypes.c_int64 * 4)(*(0 if n == 1 else s for n, s in zip(key[0], key[1])))
        _STRIDES[key] = arr
    return arr


def attn_fwd(q, k, v, out, causal, pack, block_m, block_n, qk_scale, stream):
    """Call fa2_attn_fwd on tensors that already satisfy the C contract."""
    B, H_q, N_q, D = q.shape
    H_kv, N_kv = k.shape[1], k.shape[2]
    rc = lib().fa2_attn_fwd(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
        _strides(q), _strides(k), _strides(v), _strides(out),
        B, H_q, H_kv, N_q, N_kv, D, DTYPE_CODE[q.dtype], int(bool(causal)), pack,
        block_m, block_n, qk_scale, stream)
    if rc != 0:
        raise RuntimeError(f"fa2_attn_fwd failed ({rc}): {last_error()}")


def attn_fwd_ex(q, k, v, out, causal, pack, block_m, block_n, qk_scale, lse, num_splits,
                workspace, stream):
    """Call fa2_attn_fwd_ex: lse (fp32 [B, H_q, N_q]) and workspace (uint8) may be None."""
    B, H_q, N_q, D = q.shape
    H_kv, N_kv = k.shape[1], k.shape[2]
    rc = lib().fa2_attn_fwd_ex(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
        _strides(q), _strides(k), _strides(v), _strides(out),
        B, H_q, H_kv, N_q, N_kv, D, DTYPE_CODE[q.dtype], int(bool(causal)), pack,
        block_m, block_n, qk_scale, None if lse is None else lse.data_ptr(), num_splits,
        None if workspace is None else workspace.data_ptr(),
        0 if workspace is None else workspace.numel(), stream)
    if rc != 0:
        raise RuntimeError(f"fa2_attn_fwd_ex failed ({rc}): {last_error()}")


def attn_fwd_noalloc(q, k, v, out, causal, pack, block_m, block_n, qk_scale, lse, num_splits,
                     stream):
    """Call fa2_attn_fwd_noalloc: fa2_attn_fwd_ex with the library's own scratch as the
    workspace (no allocation anywhere); lse (fp32 [B, H_q, N_q]) may be None."""
    B, H_q, N_q, D = q.shape
    H_kv, N_kv = k.shape[1], k.shape[2]
    rc = lib().fa2_attn_fwd_noalloc(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
        _strides(q), _strides(k), _strides(v), _strides(out),
        B, H_q, H_kv, N_q, N_kv, D, DTYPE_CODE[q.dtype], int(bool(causal)), pack,
        block_m, block_n, qk_scale, None if lse is None else lse.data_ptr(), num_splits, stream)
    if rc != 0:
        raise RuntimeError(f"fa2_attn_fwd_noalloc failed ({rc}): {last_error()}")


def workspace_bytes(B, H_q, N_q, D, num_splits):
    return int(lib().fa2_workspace_bytes(B, H_q, N_q, D, num_splits))


_WS_FOR = {}


def workspace_bytes_for(B, H_q, H_kv, N_q, N_kv, D, dtype, causal, num_splits):
    """fa2_workspace_bytes_for, cached per shape (it is host policy, a pure function)."""
    key = (B, H_q, H_kv, N_q, N_kv, D, dtype, bool(causal), num_splits)
    n = _WS_FOR.get(key)
    if n is None:
        if len(_WS_FOR) >= 1024:
            _WS_FOR.clear()
        n = int(lib().fa2_workspace_bytes_for(B, H_q, H_kv, N_q, N_kv, D, DTYPE_CODE[dtype],
                                              int(bool(causal)), num_splits))
        _WS_FOR[key] = n
    return n


def num_splits(B, H_q, H_kv, N_q, N_kv, D, causal, block_m, block_n, num_cus):
    return int(lib().fa2_num_splits(B, H_q, H_kv, N_q, N_kv, D, int(bool(causal)), block_m,
                                    block_n, num_cus))
