"""Encoder layers as single library calls, for forwards bound by the host.

Run op by op, a layer of few tokens costs about 80 us of Python (argument checks,
allocations, seven library calls) for 45 us of kernels.  :class:`NativeLayer` hands the
layer's pointers to ``dflash_encoder_layer_fwd``, which launches the same kernels in the
same order.  Pointers, shapes and dtypes are read from the modules on every call, so
replaced parameters are seen; anything the call does not cover returns ``None`` and the
layer runs op by op.
"""

from __future__ import annotations

import ctypes

import torch
from torch import nn

from . import _lib, layers
from .kernel import (
    SUPPORTED_HEAD_DIMS,
    HipInferenceDisentangledSelfAttention,
    HipPreparedPositionPlan,
)

# Rows (tokens) up to which an eager forward is bound by the host: from here a layer's
# kernels take longer than its Python, and op by op its intermediates are freed earlier.
MAX_ROWS = 4096


_Attention = HipInferenceDisentangledSelfAttention
_FORWARD_PREPARED = _Attention.forward_prepared
_FUSED_PROJECTION = _Attention._fused_projection


def _runs_as_written(attention: nn.Module) -> bool:
    """False where a subclass or the instance overrides what the library call stands for."""

    state = attention.__dict__
    return type(attention) is _Attention and _Attention.forward_prepared is _FORWARD_PREPARED \
        and _Attention._fused_projection is _FUSED_PROJECTION \
        and "forward_prepared" not in state and "_fused_projection" not in state


def _taken(weight: torch.Tensor | None, bias: torch.Tensor | None, dtype: torch.dtype,
           device: int, shape: tuple[int, ...]) -> bool:
    """True if the library takes a weight of ``shape`` and its bias: one dtype, one device,
    dense."""

    return (weight is not None and bias is not None
            and weight.dtype is dtype and bias.dtype is dtype
            and weight.shape == shape and bias.shape == shape[:1]
            and weight.get_device() == device and bias.get_device() == device
            and weight.is_contiguous() and bias.is_contiguous())


class NativeLayer:
    """One layer of an encoder program whose tails and intermediate are all fused."""

    def __init__(self, attention: HipInferenceDisentangledSelfAttention,
                 attention_output: nn.Module, intermediate: nn.Module, output: nn.Module) -> None:
        self.attention = attention
        self.attention_output = attention_output
        self.intermediate = intermediate
        self.output = output

    def describe(self, x: torch.Tensor, plan: HipPreparedPositionPlan) -> _lib.EncoderLayer | None:
        """The call's layer description, or ``None`` where the layer runs op by op."""

        attention = self.attention
        prep = attention._prepared
        if prep is None or attention.relative_mode != "fused" or not _runs_as_written(attention) \
                or not layers.intermediate_is_dense_gelu(self.intermediate):
            return None
        dtype, device, (_, length, hidden) = x.dtype, x.get_device(), x.shape
        heads, dim = attention.num_attention_heads, attention.attention_head_size
        width = heads * dim
        inner_dense = self.intermediate._modules["dense"]
        inner = inner_dense.out_features
        # (gemm_width_fits of the four projections: their K are multiples of 32 where the
        # columns of the others fit and the head dimension is one of these.)
        if dim not in SUPPORTED_HEAD_DIMS or dtype not in layers.GEMM_DTYPES \
                or (3 * width % 128 and 3 * width % 192) or (hidden % 128 and hidden % 192) \
                or (inner % 128 and inner % 192):
            return None
        tail, last = self.attention_output._modules, self.output._modules
        attention_norm, output_norm = tail["LayerNorm"], last["LayerNorm"]
        addresses = []
        for parameters, shape in ((tail["dense"]._parameters, (hidden, width)),
                                  (attention_norm._parameters, (hidden,)),
                                  (inner_dense._parameters, (inner, hidden)),
                                  (last["dense"]._parameters, (hidden, inner)),
                                  (output_norm._parameters, (hidden,))):
            weight, bias = parameters.get("weight"), parameters.get("bias")
            if not _taken(weight, bias, dtype, device, shape):
                return None
            addresses += weight.data_ptr(), bias.data_ptr()
        qkv, qkv_bias = prep.qkv_weight, prep.qkv_bias
        if not _taken(qkv, qkv_bias, dtype, device, (3 * width, hidden)):
            return None
        qkv, qkv_bias = qkv.data_ptr(), qkv_bias.data_ptr()
        pos_key = pos_query = slots = 0
        rows = plan.pos_key
        if attention.has_c2p:
            if rows is None or rows.dtype is not dtype or rows.get_device() != device \
                    or rows.dim() != 3 or not rows.is_contiguous():
                return None
            at, slots, row = rows.shape
            if at != heads or row != dim:
                return None
            pos_key = rows.data_ptr()
        rows = plan.pos_query
        if attention.has_p2c:
            if rows is None or rows.dtype is not dtype or rows.get_device() != device \
                    or rows.dim() != 3 or not rows.is_contiguous() \
                    or rows.shape != (heads, slots or rows.size(1), dim):
                return None
            slots = rows.size(1)
            pos_query = rows.data_ptr()
        lut = plan.delta_to_local
        if lut.dtype is not torch.int32 or lut.get_device() != device \
                or lut.shape != (2 * length - 1,) or not lut.is_contiguous():
            return None
        misaligned = qkv | qkv_bias
        for at in addresses:
            misaligned |= at
        if misaligned & 15:
            return None
        return _lib.EncoderLayer.from_buffer_copy(_lib.ENCODER_LAYER_FORMAT.pack(
            qkv, qkv_bias, pos_key, pos_query, lut.data_ptr(), *addresses,
            attention.score_scale_log2(), attention_norm.eps, output_norm.eps,
            heads, dim, slots, hidden, inner, _lib.DTYPE_CODES[dtype]))


class NativeForward:
    """The layers of one forward call: one workspace, allocated when first needed."""

    def __init__(self, x: torch.Tensor, mask: torch.Tensor) -> None:
        self.lib = _lib.load()
        self.mask = mask
        self.shape = tuple(mask.shape)
        self.device = x.get_device()
        self.workspace: torch.Tensor | None = None
        self.stream = _lib.current_stream_handle(x.device)

    @staticmethod
    def covers(x: torch.Tensor, mask: torch.Tensor) -> bool:
        return (layers.USE_HIP_GEMM and layers.GEMM_CONFIG == 0 and x.dim() == 3
                and x.dtype in layers.GEMM_DTYPES and 0 < x.shape[0] * x.shape[1] <= MAX_ROWS
                and _lib.runs_directly(x)
                and type(mask) is torch.Tensor and mask.device == x.device
                and mask.shape == x.shape[:2] and mask.dtype == torch.bool
                and mask.is_contiguous())

    def run(self, layer: NativeLayer, x: torch.Tensor,
            plan: HipPreparedPositionPlan) -> torch.Tensor | None:
        # A layer's input may come from a step run op by op (the first layer's from the
        # caller, the second's from the convolution), so each is looked at; what only the
        # op-by-op path reports (training, gradients, another length) is left to it.
        if type(x) not in _lib.PLAIN_TENSORS or x.dim() != 3 or not x.is_contiguous() \
                or x.data_ptr() & 15 or x.get_device() != self.device:
            return None
        batch, length, _ = x.shape
        if (batch, length) != self.shape or length != plan.sequence_length \
                or layer.attention.training or torch.is_grad_enabled():
            return None
        described = layer.describe(x, plan)
        if described is None:
            return None
        reference = ctypes.byref(described)
        out = torch.empty_like(x)
        # The layers of a forward are mostly alike: the library says when one needs more
        # workspace (before it launches anything).
        code = _lib.ERR_WORKSPACE
        if self.workspace is not None:
            code = self.run_layer(reference, x, out)
        if code == _lib.ERR_WORKSPACE:
            size = self.lib.dflash_encoder_layer_workspace_bytes(reference, batch, length)
            if size == 0:
                return None
            self.workspace = torch.empty(size, device=x.device, dtype=torch.uint8)
            code = self.run_layer(reference, x, out)
        _lib.check(code, "dflash_encoder_layer_fwd")
        return out

    def run_layer(self, reference, x: torch.Tensor, out: torch.Tensor) -> int:
        return self.lib.dflash_encoder_layer_fwd(
            reference, x.data_ptr(), self.mask.data_ptr(), out.data_ptr(), *self.shape,
            self.workspace.data_ptr(), self.workspace.numel(), self.stream)


__all__ = ["MAX_ROWS", "NativeForward", "NativeLayer"]
