"""Fused encoder-layer tails for the HIP backend.

``DebertaV2SelfOutput`` and ``DebertaV2Output`` (reference ``_reference.py:101-112``
and ``474-485``) both end in ``LayerNorm(dense(x) + input_tensor)``.  The HIP
encoder runs the dense projection on the hand-written GEMM where
:func:`projection_on_hip` and :func:`output_on_hip` say so
(``disentangled_flash::linear_add_layernorm``), on ``F.linear`` otherwise, and replaces the
separate residual add and LayerNorm with one kernel (``disentangled_flash::add_layernorm``),
which reads the projection and the residual once and writes the normalised row.

The ``ConvLayer`` run after the first encoder layer (reference
``_reference.py:519-566``, called at ``deberta.py:272-273``) is fused the same
way: its Conv1d (kernel 3, padding 1) becomes one library GEMM of the layer
input with the three taps side by side, and one kernel,
``disentangled_flash::conv_layer_tail``, sums the taps of neighbouring rows and
applies the mask, activation, residual add, LayerNorm and output mask.

The ops have fake implementations so that ``torch.compile(fullgraph=True)``
traces through them, like the attention ops.
"""

from __future__ import annotations

import contextlib

import torch
from torch import nn
from torch.nn import functional as F
from torch.nn.modules import module as torch_module

from . import _lib


@_lib.hip_op("disentangled_flash::add_layernorm")
def add_layernorm(
    x: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor, eps: float
) -> torch.Tensor:
    """``LayerNorm(x + residual)`` over the last dimension; the sum is rounded to the dtype first."""

    lib = _lib.load()
    hidden = x.shape[-1]
    rows = x.numel() // hidden if hidden else 0
    out = torch.empty_like(x)
    code = lib.dflash_add_layernorm_fwd(
        x.data_ptr(),
        residual.data_ptr(),
        weight.data_ptr(),
        bias.data_ptr(),
        out.data_ptr(),
        rows,
        hidden,
        float(eps),
        _lib.DTYPE_CODES[x.dtype],
        _lib.current_stream_handle(x.device),
    )
    _lib.check(code, "dflash_add_layernorm_fwd")
    return out


@add_layernorm.register_fake
def _add_layernorm_fake(x, residual, weight, bias, eps):
    return torch.empty_like(x)


@_lib.hip_op("disentangled_flash::layernorm")
def layernorm(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor, eps: float) -> torch.Tensor:
    """``LayerNorm(x)`` over the last dimension (statistics in fp32)."""

    lib = _lib.load()
    hidden = x.shape[-1]
    rows = x.numel() // hidden if hidden else 0
    out = torch.empty_like(x)
    code = lib.dflash_add_layernorm_fwd(
        x.data_ptr(), None, weight.data_ptr(), bias.data_ptr(), out.data_ptr(), rows, hidden,
        float(eps), _lib.DTYPE_CODES[x.dtype], _lib.current_stream_handle(x.device))
    _lib.check(code, "dflash_add_layernorm_fwd")
    return out


@layernorm.register_fake
def _layernorm_fake(x, weight, bias, eps):
    return torch.empty_like(x)


# Whether the encoder runs its projections on the hand-written GEMM
# (dflash_linear_fwd) where it fits, or on hipBLASLt through F.linear; read when
# an encoder is prepared and on every projection.  A switch for A/B timing.
USE_HIP_GEMM = True

# Which GEMM runs an encoder projection (projection_on_hip): the hand-written one where
# it fits (gemm_fits), but the FFN output (K = 4 x hidden) from LIBRARY_FFN_OUTPUT_MIN_ROWS
# rows on hipBLASLt, which is faster there (output_on_hip).  Device times from HIP graphs
# over changing operands, hand-written / hipBLASLt (+ its GELU pass, + the fused
# add + LayerNorm for the output blocks), fp16, us, rows: QKV, attention output, FFN
# intermediate + GELU, FFN output:
#   width 768    512:   7.5 / 8.6,    9.0 / 9.7,    9.2 / 13.9,  14.0 / 16.3
#               4096:  19.5 / 20.4,  15.6 / 18.8,  24.8 / 38.6,  33.3 / 33.0
#               8192:  33.2 / 40.2,  23.0 / 25.4,  51.4 / 72.6,  50.2 / 49.9
#              12288:  51.5 / 45.8,  30.3 / 39.0,  78.2 / 99.4,  85.2 / 74.8
#              16384:  71.7 / 71.3,  37.5 / 38.7, 102.6 / 120.8, 91.3 / 84.7
#   width 1024  4096:  27.3 / 30.6,  20.0 / 22.3,  38.5 / 50.2,  46.6 / 46.2
#               8192:  54.0 / 59.6,  31.7 / 33.9,  75.7 / 91.4,  90.3 / 78.7
#              16384: 104.1 / 88.4,  52.3 / 52.4, 156.7 / 175.9, 129.7 / 121.2
#   width 1536  2048:  32.6 / 31.9,  22.3 / 23.7,  39.6 / 53.8,  55.7 / 52.6
#               4096:  57.4 / 71.6,  31.8 / 33.3,  79.3 / 98.8,  85.1 / 85.3
#               8192: 114.5 / 114.0, 50.9 / 53.1, 154.2 / 169.7, 151.7 / 139.6
# An F.linear call also costs about 19 us of hipBLASLt host time against a few.  (The QKV
# projection is behind in places too, by up to 20 %: its tiles leave a last round half
# empty.)
LIBRARY_FFN_OUTPUT_MIN_ROWS = 8192
# While torch.compile traces, the hand-written GEMM from HIP_GEMM_MIN_ROWS rows; below,
# F.linear, which Inductor fuses.  Checked on every call: the layer program binds the
# fused steps once per bucket, while B varies per call.
HIP_GEMM_MIN_ROWS = 16384


@contextlib.contextmanager
def graph_gemm_choice():
    """For callers that compare with a captured bucket: eager forwards run the GEMMs that a
    capture records, bit for bit, inside this block and outside it."""

    yield


def projection_on_hip(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None) -> bool:
    """True if ``F.linear(x, weight, bias)`` runs on the hand-written GEMM, by the rules
    above and by the operands as they lie now (parameters may have been replaced since
    the encoder was prepared); everything else stays on ``F.linear``."""

    if not USE_HIP_GEMM or x.device.type != "cuda" or x.dim() == 0 \
            or not gemm_fits(weight, bias) or x.dtype != weight.dtype \
            or x.shape[-1] != weight.shape[1] or x.device != weight.device:
        return False
    if torch.compiler.is_compiling():
        return x.numel() // x.shape[-1] >= HIP_GEMM_MIN_ROWS
    n, k = weight.shape
    if x.numel() // k * max(n, k) >= GEMM_MAX_ELEMENTS:
        return False
    # (x is copied where it lies askew, gemm_rows; without plain tensors there is no address
    # to look at, and the op's dispatch decides.)
    return not _lib.runs_directly(weight) \
        or (weight.data_ptr() % 16 == 0 and bias.data_ptr() % 8 == 0)


def output_on_hip(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None) -> bool:
    """:func:`projection_on_hip` for the projection of an output block, whose FFN form (``K``
    at least twice ``N``) of many rows stays on ``F.linear``."""

    n, k = weight.shape
    if k >= 2 * n and k > 0 and x.numel() // k >= LIBRARY_FFN_OUTPUT_MIN_ROWS:
        return False
    return projection_on_hip(x, weight, bias)


# Tile configuration the encoder asks dflash_linear_fwd for (bits 8.. of its
# epilogue argument; 0 = the library's choice by shape).  A switch for A/B timing.
GEMM_CONFIG = 0

# dflash_linear_fwd epilogues.
GEMM_BIAS = 0
GEMM_BIAS_GELU = 1
GEMM_BIAS_ADD = 2
GEMM_DTYPES = (torch.float16, torch.bfloat16)
GEMM_MAX_ELEMENTS = 1 << 31  # of x and of the output (dflash_linear_fwd takes fewer)


@_lib.hip_op("disentangled_flash::linear_epilogue")
def linear_epilogue(
    x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor, residual: torch.Tensor | None,
    epilogue: int
) -> torch.Tensor:
    """``epilogue(x @ weight.T + bias)`` on the hand-written gfx950 GEMM.

    ``x`` is ``[..., K]`` with dense rows, ``weight`` the ``[N, K]`` nn.Linear
    weight; epilogue ``GEMM_BIAS`` (plain linear), ``GEMM_BIAS_GELU`` (exact-erf
    GELU of the dtype-rounded linear output) or ``GEMM_BIAS_ADD`` (plus
    ``residual`` ``[..., N]``, after rounding the linear output).
    """

    lib = _lib.load()
    k = x.shape[-1]
    n = weight.shape[0]
    rows = x.numel() // k if k else 0
    out = x.new_empty(x.shape[:-1] + (n,))
    if int(epilogue) == GEMM_BIAS_ADD:
        # The kernel reads rows * n elements of the residual in the output dtype.
        if residual is None:
            raise ValueError("linear_epilogue: GEMM_BIAS_ADD needs a residual")
        if residual.shape != out.shape:
            raise ValueError(f"linear_epilogue: residual shape {tuple(residual.shape)} "
                             f"!= output shape {tuple(out.shape)}")
        if residual.dtype != x.dtype or residual.device != x.device:
            raise ValueError("linear_epilogue: residual must have the input's dtype and device")
        if not residual.is_contiguous():
            raise ValueError("linear_epilogue: residual must be contiguous")
    code = lib.dflash_linear_fwd(
        x.data_ptr(), weight.data_ptr(), bias.data_ptr(),
        residual.data_ptr() if residual is not None else None, out.data_ptr(), rows, n, k,
        int(epilogue) | (int(GEMM_CONFIG) << 8), _lib.DTYPE_CODES[x.dtype],
        _lib.current_stream_handle(x.device))
    _lib.check(code, "dflash_linear_fwd")
    return out


@linear_epilogue.register_fake
def _linear_epilogue_fake(x, weight, bias, residual, epilogue):
    return x.new_empty(x.shape[:-1] + (weight.shape[0],))


@_lib.hip_op("disentangled_flash::linear_add_layernorm")
def linear_add_layernorm(
    x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor, residual: torch.Tensor,
    norm_weight: torch.Tensor, norm_bias: torch.Tensor, eps: float
) -> torch.Tensor:
    """``LayerNorm(x @ weight.T + bias + residual)``: the hand-written GEMM, then the fused
    add + LayerNorm, which for few rows also adds the GEMM's K ranges."""

    lib = _lib.load()
    k = x.shape[-1]
    n = weight.shape[0]
    rows = x.numel() // k if k else 0
    if residual.shape[-1] != n or residual.numel() != rows * n or residual.dtype != x.dtype \
            or residual.device != x.device or not residual.is_contiguous():
        raise ValueError("linear_add_layernorm: residual must be contiguous [..., N] of the "
                         "input's rows, dtype and device")
    out = x.new_empty(x.shape[:-1] + (n,))
    size = lib.dflash_output_block_workspace_bytes(rows, n, k)
    workspace = torch.empty(size, device=x.device, dtype=torch.uint8)
    code = lib.dflash_output_block_fwd(
        x.data_ptr(), weight.data_ptr(), bias.data_ptr(), residual.data_ptr(),
        norm_weight.data_ptr(), norm_bias.data_ptr(), out.data_ptr(), rows, n, k, float(eps),
        _lib.DTYPE_CODES[x.dtype], workspace.data_ptr(), size,
        _lib.current_stream_handle(x.device))
    _lib.check(code, "dflash_output_block_fwd")
    return out


@linear_add_layernorm.register_fake
def _linear_add_layernorm_fake(x, weight, bias, residual, norm_weight, norm_bias, eps):
    return x.new_empty(x.shape[:-1] + (weight.shape[0],))


def gemm_width_fits(n: int, k: int) -> bool:
    """True if the hand-written GEMM takes an ``[N, K]`` weight."""

    return n > 0 and (n % 128 == 0 or n % 192 == 0) and k > 0 and k % 32 == 0


def gemm_fits(weight: torch.Tensor, bias: torch.Tensor | None) -> bool:
    """True if ``F.linear(x, weight, bias)`` can run on :func:`linear_epilogue`.

    That is: fp16 or bf16 weight and bias on a GPU, contiguous, the bias of N elements, N
    a multiple of 128 or 192 (the tile widths) and K a multiple of 32 (the k-step) -
    every projection of DeBERTa base, large and xlarge.
    """

    if bias is None or weight.dim() != 2:
        return False
    n, k = weight.shape
    if weight.dtype not in GEMM_DTYPES or bias.dtype != weight.dtype:
        return False
    if not weight.is_contiguous() or weight.device.type != "cuda":
        return False
    if bias.dim() != 1 or bias.shape[0] != n or not bias.is_contiguous() \
            or bias.device != weight.device:
        return False
    return gemm_width_fits(n, k)


def linear_fits(linear: nn.Module) -> bool:
    return USE_HIP_GEMM and isinstance(linear, nn.Linear) and gemm_fits(linear.weight, linear.bias)


def gemm_rows(x: torch.Tensor) -> torch.Tensor:
    """``x`` with dense rows (last dimension contiguous, rows packed) from a 16-byte boundary."""

    if not x.is_contiguous():
        return x.contiguous()
    return x.clone() if _lib.runs_directly(x) and x.data_ptr() % 16 else x


def fusable_intermediate(module: nn.Module) -> bool:
    """True for a Hugging Face ``DebertaV2Intermediate`` whose activation is the erf GELU.

    ``dense`` must fit :func:`gemm_fits` and ``intermediate_act_fn`` must be
    transformers' ``GELUActivation`` (``ACT2FN["gelu"]``) computing the erf form,
    or ``torch.nn.functional.gelu`` itself.
    """

    return linear_fits(getattr(module, "dense", None)) \
        and _is_erf_gelu(getattr(module, "intermediate_act_fn", None))


def _is_erf_gelu(act) -> bool:
    if act is F.gelu:
        return True
    if type(act).__name__ != "GELUActivation":
        return False
    inner = getattr(act, "act", None)
    return inner is F.gelu or getattr(inner, "__name__", "") == "_gelu_python"


def intermediate_is_dense_gelu(module: nn.Module) -> bool:
    """True if calling ``module`` (a :func:`fusable_intermediate` when the encoder was prepared)
    still is its dense layer and an erf GELU: no forward hooks on any of the three or on all
    modules, no ``forward`` set on an instance, nothing replaced."""

    modules = module._modules  # (past nn.Module's attribute lookup: this runs on every call)
    dense, act = modules.get("dense"), modules.get("intermediate_act_fn")
    if act is None:
        act = module.__dict__.get("intermediate_act_fn")
    elif act._forward_hooks or act._forward_pre_hooks or "forward" in act.__dict__:
        return False
    return isinstance(dense, nn.Linear) and _is_erf_gelu(act) and not (
        module._forward_hooks or module._forward_pre_hooks or "forward" in module.__dict__
        or dense._forward_hooks or dense._forward_pre_hooks or "forward" in dense.__dict__
        or torch_module._global_forward_hooks or torch_module._global_forward_pre_hooks)


def intermediate_block(module: nn.Module, hidden_states: torch.Tensor) -> torch.Tensor:
    """``module(hidden_states)`` as one GEMM with the GELU in its epilogue, or the
    module itself where it has hooks or another activation, or where
    :func:`projection_on_hip` says so."""

    if not torch.compiler.is_compiling() and not intermediate_is_dense_gelu(module):
        return module(hidden_states)
    dense = module.dense
    weight, bias = dense.weight, dense.bias
    if not projection_on_hip(hidden_states, weight, bias):
        return module(hidden_states)
    return linear_epilogue(gemm_rows(hidden_states), weight, bias, None, GEMM_BIAS_GELU)


def fusable_output_block(module: nn.Module) -> bool:
    """True for a Hugging Face ``SelfOutput``/``Output`` block the fused tail can run.

    That is: a ``dense`` ``nn.Linear`` with bias, an affine ``nn.LayerNorm``
    over the last dimension and a ``dropout`` (the identity in inference), with
    parameters in one dtype the kernel supports.
    """

    dense = getattr(module, "dense", None)
    norm = getattr(module, "LayerNorm", None)
    if not isinstance(dense, nn.Linear) or dense.bias is None:
        return False
    if not isinstance(norm, nn.LayerNorm) or not norm.elementwise_affine or norm.bias is None:
        return False
    if len(norm.normalized_shape) != 1 or norm.normalized_shape[0] != dense.out_features:
        return False
    hidden = dense.out_features
    if hidden % 4 != 0 or hidden > 4096:
        return False
    dtype = dense.weight.dtype
    if dtype not in _lib.DTYPE_CODES or norm.weight.dtype != dtype or norm.bias.dtype != dtype:
        return False
    return hasattr(module, "dropout")


def output_block(module: nn.Module, hidden_states: torch.Tensor,
                 input_tensor: torch.Tensor) -> torch.Tensor:
    """``module(hidden_states, input_tensor)``: the dense projection, then one kernel for
    the residual add and LayerNorm.

    The residual is added there and not in the GEMM's epilogue: the same bytes, but
    the epilogue's reads stand at the end of every tile (16384 x 768 x 768: GEMM 26.3 against
    21.7 us, LayerNorm 10.8 against 13.1).  The caller checks
    :func:`fusable_output_block` once when the encoder is prepared; this function is the
    hot path.
    """

    dense = module.dense
    residual = gemm_rows(input_tensor)
    norm = module.LayerNorm
    weight, bias = dense.weight, dense.bias
    if isinstance(dense, nn.Linear) and output_on_hip(hidden_states, weight, bias):
        return linear_add_layernorm(gemm_rows(hidden_states), weight, bias, residual,
                                    norm.weight, norm.bias, norm.eps)
    projected = F.linear(hidden_states, weight, bias)
    return add_layernorm(projected, residual, norm.weight, norm.bias, norm.eps)


# ConvLayer.conv_act values the fused tail implements (DFLASH_ACT_* codes);
# "gelu" is the exact erf form of Hugging Face's ACT2FN["gelu"].
CONV_ACTIVATIONS = {"gelu": 0, "tanh": 1, "relu": 2}


@_lib.hip_op("disentangled_flash::conv_layer_tail")
def conv_layer_tail(
    taps: torch.Tensor, residual: torch.Tensor, conv_bias: torch.Tensor, weight: torch.Tensor,
    bias: torch.Tensor, mask: torch.Tensor, eps: float, act: int
) -> torch.Tensor:
    """ConvLayer output from the tap products ``taps`` ``[B*L, 3*hidden]``.

    ``residual`` is ``[B, L, hidden]``; ``mask`` the caller's ``[B, L]`` mask
    as int64 (a bool mask as 0/1).
    """

    lib = _lib.load()
    batch, length, hidden = residual.shape
    out = torch.empty_like(residual)
    code = lib.dflash_conv_layer_tail_fwd(
        taps.data_ptr(),
        _lib.DTYPE_CODES[taps.dtype],
        residual.data_ptr(),
        conv_bias.data_ptr(),
        weight.data_ptr(),
        bias.data_ptr(),
        mask.data_ptr(),
        out.data_ptr(),
        batch,
        length,
        hidden,
        float(eps),
        int(act),
        _lib.DTYPE_CODES[residual.dtype],
        _lib.current_stream_handle(residual.device),
    )
    _lib.check(code, "dflash_conv_layer_tail_fwd")
    return out


@conv_layer_tail.register_fake
def _conv_layer_tail_fake(taps, residual, conv_bias, weight, bias, mask, eps, act):
    return torch.empty_like(residual)


def fusable_conv_layer(module: nn.Module | None) -> bool:
    """True for a Hugging Face ``ConvLayer`` the fused tail can run.

    That is: ``conv`` an ``nn.Conv1d(hidden, hidden, 3, padding=1)`` with bias,
    one group, unit stride and dilation and zero padding; ``conv_act`` one of
    :data:`CONV_ACTIVATIONS`; an affine ``nn.LayerNorm`` over ``hidden``; a
    ``dropout`` (the identity in inference); one dtype the kernel supports.
    """

    if module is None:
        return False
    conv = getattr(module, "conv", None)
    norm = getattr(module, "LayerNorm", None)
    if not isinstance(conv, nn.Conv1d) or conv.bias is None:
        return False
    if (conv.kernel_size != (3,) or conv.padding != (1,) or conv.stride != (1,)
            or conv.dilation != (1,) or conv.groups != 1 or conv.padding_mode != "zeros"):
        return False
    hidden = conv.out_channels
    if conv.in_channels != hidden or hidden % 4 != 0 or hidden > 4096:
        return False
    if getattr(module, "conv_act", None) not in CONV_ACTIVATIONS:
        return False
    if not isinstance(norm, nn.LayerNorm) or not norm.elementwise_affine or norm.bias is None:
        return False
    if tuple(norm.normalized_shape) != (hidden,):
        return False
    dtype = conv.weight.dtype
    params = (conv.bias, norm.weight, norm.bias)
    if dtype not in _lib.DTYPE_CODES or any(p.dtype != dtype for p in params):
        return False
    return hasattr(module, "dropout")


def conv_taps(module: nn.Module) -> torch.Tensor:
    """Conv1d weight ``[hidden, hidden, 3]`` as ``[3*hidden, hidden]``, tap-major."""

    weight = module.conv.weight
    hidden = weight.shape[0]
    return weight.detach().permute(2, 0, 1).reshape(3 * hidden, hidden).contiguous()


def conv_layer_block(module: nn.Module, taps: torch.Tensor, hidden_states: torch.Tensor,
                     residual_states: torch.Tensor, input_mask: torch.Tensor) -> torch.Tensor:
    """``module(hidden_states, residual_states, input_mask)`` for a 2-D mask.

    The tap products are one GEMM with fp32 output for 16-bit inputs, so the
    convolution is rounded once, in the tail kernel.
    """

    batch, length, hidden = hidden_states.shape
    rows = hidden_states.reshape(batch * length, hidden)
    if hidden_states.dtype == torch.float32:
        products = torch.mm(rows, taps.t())
    else:
        products = torch.ops.aten.mm.dtype(rows, taps.t(), torch.float32)
    mask = input_mask if input_mask.dtype == torch.int64 else input_mask.to(torch.int64)
    residual = residual_states if residual_states.is_contiguous() else residual_states.contiguous()
    norm = module.LayerNorm
    return conv_layer_tail(products, residual, module.conv.bias, norm.weight, norm.bias,
                           mask.contiguous(), norm.eps, CONV_ACTIVATIONS[module.conv_act])


__all__ = [
    "CONV_ACTIVATIONS",
    "add_layernorm",
    "conv_layer_block",
    "conv_layer_tail",
    "conv_taps",
    "fusable_conv_layer",
    "fusable_output_block",
    "output_block",
]
