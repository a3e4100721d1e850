"""Operands that the hand-written GEMM does not take as they lie run on ``F.linear`` (or as an
aligned copy): eager forwards of few and of many tokens, and captured ones."""

from __future__ import annotations

import pytest
import torch

from test_gpu_module import _encoder_inputs, _encoder_model

pytestmark = pytest.mark.gpu

LENGTH = 64
BATCHES = (2, 80)  # 128 rows, one library call a layer, and 5120, op by op


def _encoder(dtype=torch.float16):
    from disentangled_flash import enable_deberta_inference

    return enable_deberta_inference(_encoder_model(2, 256, 4, 512).to("cuda", dtype),
                                    backend="hip", sequence_lengths=[LENGTH]).encoder


def _at_offset(values: torch.Tensor, elements: int) -> torch.Tensor:
    """The same values, contiguous, `elements` past the start of an allocation."""

    flat = torch.empty(values.numel() + elements, device=values.device, dtype=values.dtype)
    out = flat[elements:].view(values.shape)
    return out.copy_(values)


def _forward(encoder, hidden, mask):
    with torch.inference_mode():
        return encoder(hidden, mask, output_hidden_states=False).last_hidden_state


def _captured(encoder, batch, hidden, mask):
    from disentangled_flash import capture_deberta_buckets

    bucket = capture_deberta_buckets(encoder, [(batch, LENGTH)])[(batch, LENGTH)]
    return bucket(hidden, mask).clone()


def _close(got, want):
    # Two fp16 layers with another GEMM in places: LayerNorm outputs of O(1).
    assert torch.allclose(got.float(), want.float(), rtol=4e-3, atol=1.6e-2)


PARAMETERS = ("attention.output.dense", "intermediate.dense", "output.dense")


@pytest.mark.parametrize("which", ["weight", "bias", "expanded bias", "strided weight"])
@pytest.mark.parametrize("name", PARAMETERS)
def test_replaced_parameters(name, which):
    encoder = _encoder()
    inputs = {}
    for batch in BATCHES:
        hidden, mask = _encoder_inputs(batch, LENGTH, 256, seed=batch)
        inputs[batch] = hidden.to("cuda", torch.float16), mask.cuda()
    dense = encoder.layer[1].get_submodule(name)
    field = which.split()[-1]
    value = getattr(dense, field).detach()
    if which == "expanded bias":  # one value read N times: stride 0
        value = value[:1].clone().expand(value.shape)
        dense.bias = torch.nn.Parameter(value.contiguous(), requires_grad=False)
    want = {batch: _forward(encoder, *inputs[batch]) for batch in BATCHES}
    if which == "strided weight":
        value = value.t().contiguous().t()
    elif which != "expanded bias":
        value = _at_offset(value, 1)
        assert value.data_ptr() % 8
    setattr(dense, field, torch.nn.Parameter(value, requires_grad=False))
    for batch in BATCHES:
        _close(_forward(encoder, *inputs[batch]), want[batch])
    _close(_captured(encoder, BATCHES[0], *inputs[BATCHES[0]]), want[BATCHES[0]])


@pytest.mark.parametrize("elements", [1, 4])
@pytest.mark.parametrize("batch", BATCHES)
def test_input_at_an_offset(batch, elements):
    encoder = _encoder()
    hidden, mask = _encoder_inputs(batch, LENGTH, 256, seed=batch)
    hidden, mask = hidden.to("cuda", torch.float16), mask.cuda()
    want = _forward(encoder, hidden, mask)
    askew = _at_offset(hidden, elements)
    assert askew.data_ptr() % 16
    _close(_forward(encoder, askew, mask), want)


def test_layer_input_that_is_not_dense():
    """The convolution's result may lie anyhow: the second layer looks at it again."""

    encoder = _encoder()
    hidden, mask = _encoder_inputs(2, LENGTH, 256, seed=5)
    hidden, mask = hidden.to("cuda", torch.float16), mask.cuda()
    fused = encoder._conv_step
    assert fused is not None
    want = _forward(encoder, hidden, mask)
    encoder.__dict__["_conv_step"] = lambda *a: fused(*a).transpose(0, 1).contiguous().transpose(0, 1)
    _close(_forward(encoder, hidden, mask), want)
    encoder.__dict__["_conv_step"] = lambda *a: _at_offset(fused(*a), 1)
    _close(_forward(encoder, hidden, mask), want)


def test_more_elements_than_the_library_takes():
    """The rule that keeps such products on ``F.linear`` , by shape alone."""

    from disentangled_flash import layers

    weight = torch.zeros(1024, 256, device="cuda", dtype=torch.float16)
    bias = torch.zeros(1024, device="cuda", dtype=torch.float16)
    row = torch.zeros(1, 256, device="cuda", dtype=torch.float16)
    assert layers.projection_on_hip(row.expand((1 << 21) - 1, 256), weight, bias)
    assert not layers.projection_on_hip(row.expand(1 << 21, 256), weight, bias)
    assert not layers.projection_on_hip(row.to(torch.bfloat16), weight, bias)
    assert not layers.projection_on_hip(row[:, :128], weight, bias)
    assert not layers.projection_on_hip(row, weight, bias[:512])
