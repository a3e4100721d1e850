"""ctypes binding of ``libdflash.so`` (the C ABI declared in ``include/dflash.h``).

The library is a plain HIP shared object built for gfx950 next to this file.
It is loaded after ``torch`` so that it binds to the HIP runtime torch already
loaded (both resolve ``libamdhip64.so.7``), which keeps torch's streams and
device pointers valid inside the library.

There is no fallback: if the library is missing or cannot be loaded, every
HIP-backend call raises ``RuntimeError``.
"""

from __future__ import annotations

import ctypes
import functools
import os
import struct
from pathlib import Path

import torch  # noqa: F401  (load torch's HIP runtime first)

LIBRARY_NAME = "libdflash.so"
ABI_VERSION = 7

ERR_WORKSPACE = -7  # DFLASH_ERR_WORKSPACE

DTYPE_CODES = {
    torch.float16: 0,
    torch.bfloat16: 1,
    torch.float32: 2,
}

_c_void_p = ctypes.c_void_p
_c_int = ctypes.c_int
_c_int64 = ctypes.c_int64
_c_float = ctypes.c_float


class EncoderLayer(ctypes.Structure):
    """``dflash_encoder_layer``: the pointers and sizes of one layer."""

    _fields_ = [(name, _c_void_p) for name in (
        "qkv_weight", "qkv_bias", "pos_key", "pos_query", "delta_to_local",
        "attention_weight", "attention_bias", "attention_gamma", "attention_beta",
        "inner_weight", "inner_bias",
        "output_weight", "output_bias", "output_gamma", "output_beta")] + [
        (name, _c_float) for name in ("score_scale_log2", "attention_eps", "output_eps")] + [
        (name, _c_int) for name in ("heads", "head_dim", "slots", "hidden", "inner", "dtype")]


# The same fields for struct.pack (a Structure takes its fields one by one, 3 us).
ENCODER_LAYER_FORMAT = struct.Struct("@15P3f6i0P")

_handle: ctypes.CDLL | None = None
_load_error: str | None = None


def library_path() -> Path:
    override = os.environ.get("DFLASH_LIBRARY")
    return Path(override) if override else Path(__file__).with_name(LIBRARY_NAME)


def _bind(lib: ctypes.CDLL) -> None:
    lib.dflash_attention_fwd.restype = _c_int
    lib.dflash_attention_fwd.argtypes = [
        _c_void_p, _c_void_p, _c_void_p,            # query, key, value
        _c_void_p, _c_void_p,                        # c2p, p2c
        _c_void_p, _c_void_p, _c_void_p,             # delta_to_local, mask, out
        _c_int, _c_int, _c_int, _c_int, _c_int,      # B, H, L, D, S
        _c_float, _c_int, _c_int, _c_int, _c_int,    # scale, has_c2p, has_p2c, dtype, strict
        _c_void_p,                                   # stream
    ]
    lib.dflash_attention_rel_fwd.restype = _c_int
    lib.dflash_attention_rel_fwd.argtypes = [
        _c_void_p, _c_void_p, _c_void_p,             # query, key, value
        _c_int64, _c_int64, _c_int64,                # stride_b, stride_h, stride_l
        _c_void_p, _c_void_p,                        # pos_key, pos_query
        _c_void_p, _c_void_p, _c_void_p,             # delta_to_local, mask, out
        _c_int, _c_int, _c_int, _c_int, _c_int,      # B, H, L, D, S
        _c_float, _c_int, _c_int, _c_int, _c_int,    # scale, has_c2p, has_p2c, dtype, strict
        _c_void_p,                                   # stream
    ]
    lib.dflash_attention_rel_split_plan.restype = _c_int
    lib.dflash_attention_rel_split_plan.argtypes = [
        _c_int, _c_int, _c_int, _c_int,                           # B, H, L, D
        ctypes.POINTER(_c_int), ctypes.POINTER(ctypes.c_size_t),  # splits, workspace_bytes
    ]
    lib.dflash_attention_rel_fwd_split.restype = _c_int
    lib.dflash_attention_rel_fwd_split.argtypes = [
        *lib.dflash_attention_rel_fwd.argtypes[:-1],              # as dflash_attention_rel_fwd
        _c_int, _c_void_p, ctypes.c_size_t,                       # splits, workspace, bytes
        _c_void_p,                                                # stream
    ]
    lib.dflash_attention_rel_fwd_noalloc.restype = _c_int
    lib.dflash_attention_rel_fwd_noalloc.argtypes = [
        *lib.dflash_attention_rel_fwd.argtypes[:-1],              # as dflash_attention_rel_fwd
        _c_int,                                                   # splits (0 = plan)
        _c_void_p,                                                # stream
    ]
    lib.dflash_attention_rel_noalloc_scratch_bytes.restype = ctypes.c_size_t
    lib.dflash_attention_rel_noalloc_scratch_bytes.argtypes = []
    lib.dflash_add_layernorm_fwd.restype = _c_int
    lib.dflash_add_layernorm_fwd.argtypes = [
        _c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p,  # x, residual, gamma, beta, out
        _c_int, _c_int, _c_float, _c_int,                        # rows, hidden, eps, dtype
        _c_void_p,                                               # stream
    ]
    lib.dflash_conv_layer_tail_fwd.restype = _c_int
    lib.dflash_conv_layer_tail_fwd.argtypes = [
        _c_void_p, _c_int,                                       # z, z_dtype
        _c_void_p, _c_void_p, _c_void_p, _c_void_p,              # residual, bias, gamma, beta
        _c_void_p, _c_void_p,                                    # mask, out
        _c_int, _c_int, _c_int, _c_float, _c_int, _c_int,        # B, L, hidden, eps, act, dtype
        _c_void_p,                                               # stream
    ]
    lib.dflash_linear_fwd.restype = _c_int
    lib.dflash_linear_fwd.argtypes = [
        _c_void_p, _c_void_p, _c_void_p, _c_void_p, _c_void_p,  # x, weight, bias, residual, y
        _c_int, _c_int, _c_int, _c_int, _c_int,                  # M, N, K, epilogue, dtype
        _c_void_p,                                               # stream
    ]
    lib.dflash_output_block_workspace_bytes.restype = ctypes.c_size_t
    lib.dflash_output_block_workspace_bytes.argtypes = [_c_int, _c_int, _c_int]  # M, N, K
    lib.dflash_output_block_fwd.restype = _c_int
    lib.dflash_output_block_fwd.argtypes = [
        _c_void_p, _c_void_p, _c_void_p, _c_void_p,              # x, weight, bias, residual
        _c_void_p, _c_void_p, _c_void_p,                         # gamma, beta, out
        _c_int, _c_int, _c_int, _c_float, _c_int,                # M, N, K, eps, dtype
        _c_void_p, ctypes.c_size_t, _c_void_p,                   # workspace, bytes, stream
    ]
    lib.dflash_encoder_layer_workspace_bytes.restype = ctypes.c_size_t
    lib.dflash_encoder_layer_workspace_bytes.argtypes = [
        ctypes.POINTER(EncoderLayer), _c_int, _c_int]            # layer, B, L
    lib.dflash_encoder_layer_fwd.restype = _c_int
    lib.dflash_encoder_layer_fwd.argtypes = [
        ctypes.POINTER(EncoderLayer), _c_void_p, _c_void_p, _c_void_p,  # layer, x, mask, out
        _c_int, _c_int,                                          # B, L
        _c_void_p, ctypes.c_size_t, _c_void_p,                   # workspace, bytes, stream
    ]
    lib.dflash_error_string.restype = ctypes.c_char_p
    lib.dflash_error_string.argtypes = [_c_int]
    lib.dflash_abi_version.restype = _c_int
    lib.dflash_abi_version.argtypes = []


def load() -> ctypes.CDLL:
    """Load and bind the library once; raise ``RuntimeError`` if it is unusable."""

    global _handle, _load_error
    if _handle is not None:
        return _handle
    path = library_path()
    if not path.exists():
        _load_error = (
            f"{path} is missing: build the HIP library first "
            "(python __graft_entry__.py, or python disentangled-flash_amd/csrc/build.py)"
        )
        raise RuntimeError(_load_error)
    try:
        lib = ctypes.CDLL(str(path))
        _bind(lib)
    except (OSError, AttributeError) as error:
        _load_error = f"cannot load {path}: {error}"
        raise RuntimeError(_load_error) from error
    version = lib.dflash_abi_version()
    if version != ABI_VERSION:
        raise RuntimeError(f"{path} has ABI version {version}, expected {ABI_VERSION}")
    _handle = lib
    return lib


def is_available() -> bool:
    try:
        load()
    except RuntimeError:
        return False
    return True


def check(code: int, what: str) -> None:
    if code != 0:
        message = load().dflash_error_string(code).decode()
        raise RuntimeError(f"{what} failed with code {code}: {message}")


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)

PLAIN_TENSORS = (torch.Tensor, torch.nn.Parameter)

try:
    from torch.utils._python_dispatch import _get_current_dispatch_mode as _get_dispatch_mode
except ImportError:  # pragma: no cover - older torch
    def _get_dispatch_mode():
        return None


def current_stream_handle(device: torch.device) -> int:
    """The HIP stream torch launches on for ``device`` (raw handle)."""

    if _raw_stream is not None:
        return _raw_stream(device.index if device.index is not None else torch.cuda.current_device())
    return torch.cuda.current_stream(device).cuda_stream


def runs_directly(tensor: torch.Tensor) -> bool:
    """True outside tracing (torch.compile, export) and dispatch modes, for a plain CUDA
    tensor: the library may be called on its address."""

    return (type(tensor) in PLAIN_TENSORS and tensor.device.type == "cuda"
            and not torch.compiler.is_compiling() and _get_dispatch_mode() is None)


def hip_op(name: str):
    """``torch.library.custom_op(name)`` whose eager calls skip the dispatcher.

    Under ``torch.compile`` tracing the function is the custom op (with the fake
    implementation registered on it), so compiled graphs keep the HIP op as one
    node.  Called eagerly - and during HIP-graph capture - it runs the
    implementation directly: the op dispatch adds about 3 us of host time per
    call, which an eager encoder forward of a few thousand tokens (bound by launch
    time) pays on every layer.
    """

    def wrap(impl):
        op = torch.library.custom_op(name, mutates_args=())(impl)

        @functools.wraps(impl)
        def call(*args, **kwargs):
            # Through the custom op when tracing (torch.compile, export,
            # make_fx), under any dispatch mode (FakeTensorMode, opcheck) or
            # with a tensor that is not a plain CUDA tensor, so that the
            # registered fake runs instead of a data_ptr() of a fake tensor.
            if torch.compiler.is_compiling() or _get_dispatch_mode() is not None:
                return op(*args, **kwargs)
            for a in args:
                if isinstance(a, torch.Tensor) and (
                        type(a) not in PLAIN_TENSORS or a.device.type != "cuda"):
                    return op(*args, **kwargs)
            return impl(*args, **kwargs)

        call.register_fake = op.register_fake
        call.custom_op = op
        return call

    return wrap


__all__ = ["DTYPE_CODES", "check", "current_stream_handle", "hip_op", "is_available",
           "library_path", "load"]
