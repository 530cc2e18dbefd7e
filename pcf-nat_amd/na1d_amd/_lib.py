"""ctypes binding of libna1d.so (the C ABI declared in include/na1d.h).

The library is prebuilt in-tree (``pcf-nat_amd/lib/libna1d.so``); nothing is
compiled at import.  There is no CPU fallback: if the library is missing or a
call fails, a Python exception is raised.
"""
from __future__ import annotations

import ctypes
import importlib.util
import os

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.environ.get("NA1D_LIB") or os.path.join(os.path.dirname(_HERE), "lib", "libna1d.so")   # NA1D_LIB: another build

BF16, FP16 = 0, 1

_i64, _int, _f32, _ptr, _u64 = ctypes.c_int64, ctypes.c_int, ctypes.c_float, ctypes.c_void_p, ctypes.c_uint64

_UNFUSED = ("na1d_qk_forward", "na1d_av_forward", "na1d_q_backward", "na1d_k_backward",
            "na1d_a_backward", "na1d_v_backward")
SYMBOLS = _UNFUSED + ("na1d_fused_forward", "na1d_fused_backward", "na1d_fused_backward_workspace_bytes",
                      "na1d_fused_forward_strided", "na1d_fused_backward_strided", "na1d_profile_events",
                      "na1d_global_forward", "na1d_global_backward", "na1d_global_backward_workspace_bytes",
                      "na1d_fused_forward_dropout", "na1d_fused_backward_dropout",
                      "na1d_fused_backward_noalloc", "na1d_force_generic", "na1d_profile_last_kernel",
                      "na1d_fused_forward_strided_dropout", "na1d_fused_backward_strided_dropout",
                      "na1d_fused_forward_dilated", "na1d_fused_forward_clear", "na1d_fused_backward_dilated",
                      "na1d_fused_backward_dilated_workspace_bytes", "na1d_encode", "na1d_encode_workspace_bytes",
                      "na1d_train_layer_saved_bytes", "na1d_train_layer_workspace_bytes", "na1d_train_layer_forward",
                      "na1d_train_to_channels", "na1d_train_pool_backward", "na1d_train_context_backward", "na1d_train_context",
                      "na1d_train_layer_backward", "na1d_version", "na1d_status_string")
UNSUPPORTED = -8

_lib = None
_nodes = None
_other_build = "NA1D_LIB" in os.environ


class NA1DError(RuntimeError):
    """A libna1d entry point returned a non-zero status."""


def build_hint() -> str:
    return ("libna1d.so not found at %s - build it with `make -C pcf-nat_amd/csrc` "
            "(or `python -c 'import __graft_entry__ as g; g.build()'`)" % LIB_PATH)


def load():
    """Load (once) and return the ctypes handle; raises if the library is absent."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise NA1DError(build_hint())
    lib = ctypes.CDLL(LIB_PATH)
    for name in _UNFUSED:
        f = getattr(lib, name)
        f.restype = _int
        f.argtypes = [_ptr, _ptr, _ptr, _i64, _i64, _i64, _i64, _i64, _int, _ptr]
    lib.na1d_fused_forward.restype = _int
    lib.na1d_fused_forward.argtypes = [_ptr, _ptr, _ptr, _ptr, _ptr, _ptr, _ptr,
                                       _i64, _i64, _i64, _i64, _i64, _i64, _f32, _int, _ptr]
    lib.na1d_fused_backward.restype = _int
    lib.na1d_fused_backward.argtypes = [_ptr] * 12 + [_i64] * 6 + [_f32, _int, _ptr, _i64, _ptr]
    lib.na1d_fused_forward_strided.restype = _int
    lib.na1d_fused_forward_strided.argtypes = [_ptr] * 7 + [_i64] * 6 + [_f32, _int, _ptr, _ptr, _ptr]
    lib.na1d_fused_backward_strided.restype = _int
    lib.na1d_fused_backward_strided.argtypes = [_ptr] * 11 + [_i64] * 6 + [_f32, _int, _ptr, _ptr, _ptr, _i64, _ptr]
    lib.na1d_fused_backward_workspace_bytes.restype = _i64
    lib.na1d_fused_backward_workspace_bytes.argtypes = [_i64] * 6 + [_int]
    lib.na1d_fused_forward_dropout.restype = _int
    lib.na1d_fused_forward_dropout.argtypes = [_ptr] * 7 + [_i64] * 6 + [_f32, _int, _f32, _u64, _ptr]
    lib.na1d_fused_backward_dropout.restype = _int
    lib.na1d_fused_backward_dropout.argtypes = [_ptr] * 12 + [_i64] * 6 + [_f32, _int, _f32, _u64, _ptr, _i64, _ptr]
    lib.na1d_global_forward.restype = _int
    lib.na1d_global_forward.argtypes = [_ptr] * 6 + [_i64] * 4 + [_f32, _int, _f32, _u64, _ptr]
    lib.na1d_global_backward.restype = _int
    lib.na1d_global_backward.argtypes = [_ptr] * 10 + [_i64] * 4 + [_f32, _int, _f32, _u64, _ptr, _i64, _ptr]
    lib.na1d_global_backward_workspace_bytes.restype = _i64
    lib.na1d_global_backward_workspace_bytes.argtypes = [_i64] * 4 + [_int]
    lib.na1d_fused_forward_strided_dropout.restype = _int
    lib.na1d_fused_forward_strided_dropout.argtypes = [_ptr] * 7 + [_i64] * 6 + [_f32, _int, _ptr, _ptr, _f32, _u64,
                                                                              _i64, _i64, _i64, _ptr]
    lib.na1d_fused_backward_strided_dropout.restype = _int
    lib.na1d_fused_backward_strided_dropout.argtypes = [_ptr] * 11 + [_i64] * 6 + [_f32, _int, _ptr, _ptr, _f32, _u64,
                                                                                _i64, _i64, _i64, _ptr, _i64, _ptr]
    lib.na1d_fused_forward_dilated.restype = _int
    lib.na1d_fused_forward_dilated.argtypes = [_ptr] * 7 + [_i64] * 7 + [_f32, _int, _ptr, _ptr, _f32, _u64, _ptr]
    lib.na1d_fused_forward_clear.restype = _int
    lib.na1d_fused_forward_clear.argtypes = [_ptr] * 8 + [_i64] * 7 + [_f32, _int, _ptr, _ptr, _f32, _u64, _ptr]
    lib.na1d_fused_backward_dilated.restype = _int
    lib.na1d_fused_backward_dilated.argtypes = [_ptr] * 11 + [_i64] * 7 + [_f32, _int, _ptr, _ptr, _f32, _u64, _ptr, _i64,
                                                                          _ptr]
    lib.na1d_fused_backward_dilated_workspace_bytes.restype = _i64
    lib.na1d_fused_backward_dilated_workspace_bytes.argtypes = [_i64] * 7 + [_int]
    lib.na1d_encode_workspace_bytes.restype = _i64
    lib.na1d_encode_workspace_bytes.argtypes = [_ptr, _i64, _i64]
    lib.na1d_encode.restype = _int
    lib.na1d_encode.argtypes = [_ptr] * 4 + [_i64, _i64, _ptr, _i64, _ptr]
    lib.na1d_train_layer_saved_bytes.restype = lib.na1d_train_layer_workspace_bytes.restype = _i64
    lib.na1d_train_layer_saved_bytes.argtypes = [_ptr, _i64, _i64]
    lib.na1d_train_layer_workspace_bytes.argtypes = [_ptr, _i64, _i64, _int]
    lib.na1d_train_layer_forward.restype = lib.na1d_train_layer_backward.restype = _int
    lib.na1d_train_layer_forward.argtypes = [_ptr, _int] + [_ptr] * 3 + [_i64, _ptr, _i64, _i64, _i64, _ptr]
    lib.na1d_train_to_channels.restype = _int
    lib.na1d_train_to_channels.argtypes = [_ptr] * 3 + [_i64, _i64, _ptr]
    lib.na1d_train_context.restype = _int
    lib.na1d_train_context.argtypes = [_ptr] * 4 + [_i64] * 3 + [_ptr]
    lib.na1d_train_pool_backward.restype = lib.na1d_train_context_backward.restype = _int
    lib.na1d_train_pool_backward.argtypes = [_ptr] * 6 + [_i64] * 3 + [_f32, _int, _ptr]
    lib.na1d_train_context_backward.argtypes = [_ptr] * 5 + [_i64] * 3 + [_f32, _int, _ptr]
    lib.na1d_train_layer_backward.argtypes = [_ptr] * 5 + [_i64, _ptr, _i64, _i64, _i64, _ptr]
    lib.na1d_fused_backward_noalloc.restype = _int
    lib.na1d_fused_backward_noalloc.argtypes = [_ptr] * 12 + [_i64] * 6 + [_f32, _int, _ptr]
    lib.na1d_force_generic.restype = _int
    lib.na1d_force_generic.argtypes = [_int]
    lib.na1d_profile_events.restype = _int
    lib.na1d_profile_events.argtypes = [_ptr, _ptr]
    lib.na1d_profile_last_kernel.restype = ctypes.c_char_p
    lib.na1d_profile_last_kernel.argtypes = []
    lib.na1d_version.restype = _int
    lib.na1d_version.argtypes = []
    lib.na1d_status_string.restype = ctypes.c_char_p
    lib.na1d_status_string.argtypes = [_int]
    _lib = lib
    return lib


def nodes():
    """The operators' autograd nodes in C++ (``csrc/na1d_torch.cpp``).  They call the library beside them: with
    another build named by NA1D_LIB, and under ``torch.compile``, the Python implementations serve (``None``)."""
    global _nodes
    if _other_build or torch.compiler.is_compiling():
        return None
    if _nodes is None:
        load()
        path = os.path.join(os.path.dirname(LIB_PATH), "na1d_torch.so")
        if not os.path.exists(path):
            raise NA1DError(build_hint().replace(LIB_PATH, path).replace("libna1d.so", "na1d_torch.so"))
        spec = importlib.util.spec_from_file_location("na1d_torch", path)
        module = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(module)
        module.raise_as(NA1DError)
        _nodes = module
    return _nodes


def dtype_tag(dtype: torch.dtype) -> int:
    if dtype == torch.bfloat16:
        return BF16
    if dtype == torch.float16:
        return FP16
    raise TypeError("NA1D supports torch.bfloat16 and torch.float16, got %s" % dtype)


def _stream(t: torch.Tensor):
    if t.device.type != "cuda":
        raise NA1DError("NA1D tensors must live on the GPU (got device %s); there is no CPU path" % t.device)
    return ctypes.c_void_p(torch.cuda.current_stream(t.device).cuda_stream)


def _p(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def check(status: int, name: str):
    if status != 0:
        raise NA1DError("%s failed: %s (status %d)" % (name, load().na1d_status_string(status).decode(), status))


def call_unfused(name: str, out, a, b, B, T, C, W, left, dtype):
    """``name(out, a, b, B, T, C, W, left, dtype, stream)`` on torch's current stream."""
    lib = load()
    with torch.cuda.device(out.device):
        st = getattr(lib, name)(_p(out), _p(a), _p(b), B, T, C, W, left, dtype_tag(dtype), _stream(out))
    check(st, name)


def call_fused_forward(out, lse, q, k, v, rpb, t_valid, B, H, T, C, W, left, scale, dropout=None):
    """``dropout``: ``None`` or ``(p, seed)`` for the entry point with attention dropout."""
    lib = load()
    with torch.cuda.device(out.device):
        if dropout is None:
            st = lib.na1d_fused_forward(_p(out), _p(lse), _p(q), _p(k), _p(v), _p(rpb), _p(t_valid),
                                        B, H, T, C, W, left, scale, dtype_tag(q.dtype), _stream(out))
        else:
            st = lib.na1d_fused_forward_dropout(_p(out), _p(lse), _p(q), _p(k), _p(v), _p(rpb), _p(t_valid), B, H, T,
                                                C, W, left, scale, dtype_tag(q.dtype), dropout[0], dropout[1],
                                                _stream(out))
    check(st, "na1d_fused_forward")


def fused_backward_workspace_bytes(B, H, T, C, W, left, dtype) -> int:
    n = load().na1d_fused_backward_workspace_bytes(B, H, T, C, W, left, dtype_tag(dtype))
    if n < 0:
        check(int(n), "na1d_fused_backward_workspace_bytes")
    return int(n)


def call_fused_backward(dq, dk, dv, drpb, q, k, v, out, dout, lse, rpb, t_valid, B, H, T, C, W, left, scale,
                        workspace=None, dropout=None):
    """``workspace``: optional uint8/any CUDA tensor used for the d rpb reduction; ``dropout`` as in the forward."""
    lib = load()
    ws_bytes = 0 if workspace is None else workspace.numel() * workspace.element_size()
    with torch.cuda.device(dq.device):
        if dropout is None:
            st = lib.na1d_fused_backward(_p(dq), _p(dk), _p(dv), _p(drpb), _p(q), _p(k), _p(v), _p(out), _p(dout),
                                         _p(lse), _p(rpb), _p(t_valid), B, H, T, C, W, left, scale,
                                         dtype_tag(q.dtype), _p(workspace), ws_bytes, _stream(dq))
        else:
            st = lib.na1d_fused_backward_dropout(_p(dq), _p(dk), _p(dv), _p(drpb), _p(q), _p(k), _p(v), _p(out),
                                                 _p(dout), _p(lse), _p(rpb), _p(t_valid), B, H, T, C, W, left, scale,
                                                 dtype_tag(q.dtype), dropout[0], dropout[1], _p(workspace), ws_bytes,
                                                 _stream(dq))
    check(st, "na1d_fused_backward")


def _strides3(view):
    """{sample, head, row} element strides of a ``[N, H, T, C]`` view with contiguous channels."""
    assert view.dim() == 4 and (view.shape[3] == 1 or view.stride(3) == 1), "channels must be contiguous"
    return (_i64 * 3)(view.stride(0), view.stride(1), view.stride(2))


def call_fused_forward_strided(out, lse, q, k, v, rpb, t_valid, W, left, scale, dropout=None):
    """q, k, v, out: ``[N, H, T, C]`` views (q, k, v with equal strides).  Returns the status so that the
    caller can pack the tensors when no strided kernel covers the shape (``UNSUPPORTED``).  ``dropout``: ``None`` or
    ``(p, seed, row_stride, row_offset, seq_rows)`` - see na1d_fused_forward_strided_dropout."""
    lib = load()
    N, H, T, C = q.shape
    assert q.stride() == k.stride() == v.stride()
    with torch.cuda.device(out.device):
        if dropout is None:
            st = lib.na1d_fused_forward_strided(_p(out), _p(lse), _p(q), _p(k), _p(v), _p(rpb), _p(t_valid), N, H, T, C,
                                                W, left, scale, dtype_tag(q.dtype), _strides3(q), _strides3(out),
                                                _stream(out))
        else:
            st = lib.na1d_fused_forward_strided_dropout(_p(out), _p(lse), _p(q), _p(k), _p(v), _p(rpb), _p(t_valid), N,
                                                        H, T, C, W, left, scale, dtype_tag(q.dtype), _strides3(q),
                                                        _strides3(out), *dropout, _stream(out))
    if st != UNSUPPORTED:
        check(st, "na1d_fused_forward_strided")
    return st


def call_fused_backward_strided(dq, dk, dv, drpb, q, k, v, dout, lse, rpb, t_valid, W, left, scale, workspace=None,
                                dropout=None):
    lib = load()
    N, H, T, C = q.shape
    assert q.stride() == k.stride() == v.stride() == dq.stride() == dk.stride() == dv.stride()
    ws_bytes = 0 if workspace is None else workspace.numel() * workspace.element_size()
    with torch.cuda.device(dq.device):
        if dropout is None:
            st = lib.na1d_fused_backward_strided(_p(dq), _p(dk), _p(dv), _p(drpb), _p(q), _p(k), _p(v), _p(dout),
                                                 _p(lse), _p(rpb), _p(t_valid), N, H, T, C, W, left, scale,
                                                 dtype_tag(q.dtype), _strides3(q), _strides3(dout), _p(workspace),
                                                 ws_bytes, _stream(dq))
        else:
            st = lib.na1d_fused_backward_strided_dropout(_p(dq), _p(dk), _p(dv), _p(drpb), _p(q), _p(k), _p(v),
                                                         _p(dout), _p(lse), _p(rpb), _p(t_valid), N, H, T, C, W, left,
                                                         scale, dtype_tag(q.dtype), _strides3(q), _strides3(dout),
                                                         *dropout, _p(workspace), ws_bytes, _stream(dq))
    if st != UNSUPPORTED:
        check(st, "na1d_fused_backward_strided")
    return st


def call_fused_forward_dilated(out, lse, q, k, v, rpb, t_valid, W, left, dilation, scale, dropout=None):
    """All residue classes of a dilated window in one launch, on ``[N, H, T, C]`` views as in
    :func:`call_fused_forward_strided`.  ``dropout``: ``None`` or ``(p, seed)``."""
    lib = load()
    N, H, T, C = q.shape
    assert q.stride() == k.stride() == v.stride()
    with torch.cuda.device(out.device):
        st = lib.na1d_fused_forward_dilated(_p(out), _p(lse), _p(q), _p(k), _p(v), _p(rpb), _p(t_valid), N, H, T, C, W,
                                            left, dilation, scale, dtype_tag(q.dtype), _strides3(q), _strides3(out),
                                            *(dropout or (0.0, 0)), _stream(out))
    if st != UNSUPPORTED:
        check(st, "na1d_fused_forward_dilated")
    return st


def call_fused_backward_dilated(dq, dk, dv, drpb, q, k, v, dout, lse, rpb, t_valid, W, left, dilation, scale,
                                workspace=None, dropout=None):
    lib = load()
    N, H, T, C = q.shape
    assert q.stride() == k.stride() == v.stride() == dq.stride() == dk.stride() == dv.stride()
    ws_bytes = 0 if workspace is None else workspace.numel() * workspace.element_size()
    with torch.cuda.device(dq.device):
        st = lib.na1d_fused_backward_dilated(_p(dq), _p(dk), _p(dv), _p(drpb), _p(q), _p(k), _p(v), _p(dout), _p(lse),
                                             _p(rpb), _p(t_valid), N, H, T, C, W, left, dilation, scale,
                                             dtype_tag(q.dtype), _strides3(q), _strides3(dout), *(dropout or (0.0, 0)),
                                             _p(workspace), ws_bytes, _stream(dq))
    check(st, "na1d_fused_backward_dilated")


def fused_backward_dilated_workspace_bytes(N, H, T, C, W, left, dilation, dtype) -> int:
    n = load().na1d_fused_backward_dilated_workspace_bytes(N, H, T, C, W, left, dilation, dtype_tag(dtype))
    if n < 0:
        check(int(n), "na1d_fused_backward_dilated_workspace_bytes")
    return int(n)


def call_global_forward(out, lse, q, k, v, t_valid, B, H, T, C, scale, dropout=None):
    """Dense attention over whole sequences; returns the status (``UNSUPPORTED`` for head_dim > 128).
    ``dropout``: ``None`` or ``(p, seed)``."""
    lib = load()
    p, seed = dropout or (0.0, 0)
    with torch.cuda.device(out.device):
        st = lib.na1d_global_forward(_p(out), _p(lse), _p(q), _p(k), _p(v), _p(t_valid), B, H, T, C, scale,
                                     dtype_tag(q.dtype), p, seed, _stream(out))
    if st != UNSUPPORTED:
        check(st, "na1d_global_forward")
    return st


def global_backward_workspace_bytes(B, H, T, C, dtype) -> int:
    n = load().na1d_global_backward_workspace_bytes(B, H, T, C, dtype_tag(dtype))
    if n < 0:
        check(int(n), "na1d_global_backward_workspace_bytes")
    return int(n)


def call_global_backward(dq, dk, dv, q, k, v, out, dout, lse, t_valid, B, H, T, C, scale, workspace, dropout=None):
    lib = load()
    p, seed = dropout or (0.0, 0)
    with torch.cuda.device(dq.device):
        st = lib.na1d_global_backward(_p(dq), _p(dk), _p(dv), _p(q), _p(k), _p(v), _p(out), _p(dout), _p(lse),
                                      _p(t_valid), B, H, T, C, scale, dtype_tag(q.dtype), p, seed, _p(workspace),
                                      workspace.numel() * workspace.element_size(), _stream(dq))
    check(st, "na1d_global_backward")


def call_fused_forward_qkv(out, lse, qkv, rpb, t_valid, W, left, scale):
    """The strided forward on a contiguous ``[N, T, 3, H, C]`` projection output, ``out`` contiguous
    ``[N, T, H*C]``: pointers and strides worked out here, without building views (the inference path's
    per-call overhead).  Returns the status like :func:`call_fused_forward_strided`."""
    lib = load()
    N, T, _, H, C = qkv.shape
    base, step = qkv.data_ptr(), H * C * qkv.element_size()
    if torch.cuda.current_device() != out.device.index:      # launches go to the device of the tensors
        with torch.cuda.device(out.device):
            return call_fused_forward_qkv(out, lse, qkv, rpb, t_valid, W, left, scale)
    st = lib.na1d_fused_forward_strided(_p(out), _p(lse), base, base + step, base + 2 * step, _p(rpb), _p(t_valid),
                                        N, H, T, C, W, left, scale, dtype_tag(qkv.dtype),
                                        (_i64 * 3)(T * 3 * H * C, C, 3 * H * C), (_i64 * 3)(T * H * C, C, H * C),
                                        _stream(out))
    if st != UNSUPPORTED:
        check(st, "na1d_fused_forward_strided")
    return st
