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


def _pointers(module: nn.Module, dtype: torch.dtype, device: torch.device,
              shape: tuple[int, ...]) -> tuple[int, int] | None:
    """Addresses of the weight (of ``shape``) and bias of an nn.Linear or nn.LayerNorm if the
    library takes them: one dtype, dense, 16-byte aligned."""

    parameters = module._parameters
    weight, bias = parameters.get("weight"), parameters.get("bias")
    if weight is None or bias is None or weight.dtype != dtype or bias.dtype != dtype \
            or weight.shape != shape or bias.shape != shape[:1] \
            or not weight.is_contiguous() or not bias.is_contiguous() \
            or weight.device != device or bias.device != device:
        return None
    at = weight.data_ptr(), bias.data_ptr()
    return at if (at[0] | at[1]) & 15 == 0 else None


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
        if prep is None or prep.qkv_bias is None or attention.relative_mode != "fused":
            return None
        dtype, device, hidden = x.dtype, x.device, x.shape[-1]
        heads, dim = attention.num_attention_heads, attention.attention_head_size
        width = heads * dim
        qkv = prep.qkv_weight
        inner_dense = self.intermediate._modules["dense"]
        inner = inner_dense.out_features
        if dim not in SUPPORTED_HEAD_DIMS or qkv.dtype != dtype or qkv.device != device \
                or qkv.shape != (3 * width, hidden) or not layers.gemm_fits(qkv, prep.qkv_bias) \
                or not layers.gemm_width_fits(hidden, width) \
                or not layers.gemm_width_fits(inner, hidden) \
                or not layers.gemm_width_fits(hidden, inner):
            return None
        tail, last = self.attention_output._modules, self.output._modules
        attention_norm, output_norm = tail["LayerNorm"], last["LayerNorm"]
        found = (_pointers(tail["dense"], dtype, device, (hidden, width)),
                 _pointers(attention_norm, dtype, device, (hidden,)),
                 _pointers(inner_dense, dtype, device, (inner, hidden)),
                 _pointers(last["dense"], dtype, device, (hidden, inner)),
                 _pointers(output_norm, dtype, device, (hidden,)))
        if None in found:
            return None
        has_c2p, has_p2c = attention.has_c2p, attention.has_p2c
        pos_key, pos_query = plan.pos_key, plan.pos_query
        slots = 0
        for rows in ((pos_key,) if has_c2p else ()) + ((pos_query,) if has_p2c else ()):
            if rows is None or rows.dtype != dtype or rows.device != device \
                    or rows.dim() != 3 or rows.size(0) != heads or rows.size(2) != dim \
                    or not rows.is_contiguous() or (slots and rows.size(1) != slots):
                return None
            slots = rows.size(1)
        lut = plan.delta_to_local
        if lut.dtype != torch.int32 or lut.device != device or lut.dim() != 1 \
                or lut.numel() != 2 * x.shape[1] - 1 or not lut.is_contiguous():
            return None
        qkv_at = qkv.data_ptr(), prep.qkv_bias.data_ptr()
        if (qkv_at[0] | qkv_at[1]) & 15:
            return None
        return _lib.EncoderLayer(
            *qkv_at,
            pos_key.data_ptr() if has_c2p else None, pos_query.data_ptr() if has_p2c else None,
            lut.data_ptr(), *found[0], *found[1], *found[2], *found[3], *found[4],
            attention.score_scale_log2(), attention_norm.eps, output_norm.eps,
            heads, dim, slots, hidden, inner, _lib.DTYPE_CODES[dtype])


class NativeForward:
    """The layers of one forward call: one workspace, allocated when first needed."""

    def __init__(self, x: torch.Tensor, mask: torch.Tensor) -> None:
        self.lib = _lib.load()
        self.mask = mask
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
        # caller, the second's from the convolution), so each is looked at.
        if x.shape[:2] != self.mask.shape or not _lib.runs_directly(x) \
                or not x.is_contiguous() or x.data_ptr() & 15:
            return None
        layer.attention._validate_hip_call(x)
        batch, length = x.shape[:2]
        if length != plan.sequence_length:
            return None  # the op-by-op path reports it
        described = layer.describe(x, plan)
        if described is None:
            return None
        reference = ctypes.byref(described)
        size = self.lib.dflash_encoder_layer_workspace_bytes(reference, batch, length)
        if size == 0:
            return None
        if self.workspace is None or self.workspace.numel() < size:
            self.workspace = torch.empty(size, device=x.device, dtype=torch.uint8)
        out = torch.empty_like(x)
        code = self.lib.dflash_encoder_layer_fwd(
            reference, x.data_ptr(), self.mask.data_ptr(), out.data_ptr(), batch, length,
            self.workspace.data_ptr(), self.workspace.numel(), self.stream)
        _lib.check(code, "dflash_encoder_layer_fwd")
        return out


__all__ = ["MAX_ROWS", "NativeForward", "NativeLayer"]
