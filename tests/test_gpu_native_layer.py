"""Encoder layers run as one library call equal the same layers run op by op, bit for bit."""

from __future__ import annotations


import pytest
import torch

from test_gpu_module import _encoder_inputs, _encoder_model

pytestmark = pytest.mark.gpu


def _forward(encoder, hidden, mask):
    with torch.inference_mode():
        return encoder(hidden, mask, output_hidden_states=True).hidden_states


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [(1, 1), (1, 16), (3, 50), (1, 512), (7, 130), (9, 512)])
def test_native_layers_equal_op_by_op(dtype, shape, monkeypatch):
    from disentangled_flash import enable_deberta_inference, native

    batch, length = shape
    model = enable_deberta_inference(_encoder_model(2, 256, 4, 512).to("cuda", dtype),
                                     backend="hip", sequence_lengths=[length])
    encoder = model.encoder
    assert all(step.native is not None for step in encoder._program)
    hidden, mask = _encoder_inputs(batch, length, 256, seed=7)
    hidden, mask = hidden.to("cuda", dtype), mask.cuda()
    calls = []
    run = native.NativeForward.run
    monkeypatch.setattr(native.NativeForward, "run",
                        lambda self, *a: calls.append(run(self, *a)) or calls[-1])
    got = _forward(encoder, hidden, mask)
    # (9, 512) is above MAX_ROWS and runs op by op anyway.
    assert len(calls) == (2 if batch * length <= native.MAX_ROWS else 0)
    assert all(out is not None for out in calls)
    monkeypatch.setattr(native, "MAX_ROWS", 0)
    want = _forward(encoder, hidden, mask)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_native_layer_sees_replaced_parameters_and_falls_back(monkeypatch):
    from disentangled_flash import enable_deberta_inference, native

    model = enable_deberta_inference(_encoder_model(2, 256, 4, 512).to("cuda", torch.float16),
                                     backend="hip", sequence_lengths=[32])
    encoder = model.encoder
    hidden, mask = _encoder_inputs(2, 32, 256, seed=3)
    hidden, mask = hidden.to("cuda", torch.float16), mask.cuda()
    before = _forward(encoder, hidden, mask)[-1]
    dense = encoder.layer[1].output.dense
    dense.weight = torch.nn.Parameter(dense.weight * 2, requires_grad=False)
    after = _forward(encoder, hidden, mask)[-1]
    assert not torch.equal(before, after)
    # A weight the library does not take as it lies (not contiguous): op by op, same values.
    strided = torch.empty(512, 256, device="cuda", dtype=torch.float16).t()
    strided.copy_(dense.weight)
    dense.weight = torch.nn.Parameter(strided, requires_grad=False)
    assert torch.allclose(_forward(encoder, hidden, mask)[-1].float(), after.float(),
                          rtol=2e-3, atol=4e-3)
    # Another mask type, a strided input: converted as before.
    assert torch.equal(_forward(encoder, hidden, mask.bool())[0], hidden)
    wide = torch.empty(2, 32, 512, device="cuda", dtype=torch.float16)[..., :256]
    wide.copy_(hidden)
    assert _forward(encoder, wide, mask)[-1].shape == (2, 32, 256)
    with pytest.raises(ValueError):
        _forward(encoder, hidden[:, :16], mask[:, :16])
    with torch.enable_grad(), pytest.raises(RuntimeError):
        encoder(hidden, mask)


def test_encoder_layer_refusals():
    from ctypes import byref

    from disentangled_flash import _lib, enable_deberta_inference
    from disentangled_flash.native import NativeForward

    lib = _lib.load()
    model = enable_deberta_inference(_encoder_model(1, 256, 4, 512).to("cuda", torch.float16),
                                     backend="hip", sequence_lengths=[32])
    encoder = model.encoder
    x = torch.randn(2, 32, 256, device="cuda").half()
    mask = torch.ones(2, 32, device="cuda", dtype=torch.bool)
    assert NativeForward.covers(x, mask) and not NativeForward.covers(x.float(), mask)
    layer = encoder._program[0].native.describe(x, encoder.active_plans[0])
    size = lib.dflash_encoder_layer_workspace_bytes(byref(layer), 2, 32)
    ws = torch.empty(size, device="cuda", dtype=torch.uint8)
    out = torch.empty_like(x)
    stream = torch.cuda.current_stream().cuda_stream

    def call(description, batch=2, workspace=ws.data_ptr(), bytes_=size, source=x.data_ptr()):
        return lib.dflash_encoder_layer_fwd(byref(description), source, mask.data_ptr(),
                                            out.data_ptr(), batch, 32, workspace, bytes_, stream)

    assert call(layer) == 0 and call(layer, batch=0) == 0
    assert call(layer, bytes_=size - 1) == -7
    assert call(layer, workspace=None) == -1 and call(layer, source=None) == -1
    for field, value, code in (("dtype", 2, -4), ("head_dim", 48, -3), ("heads", 0, -2)):
        changed = _lib.EncoderLayer.from_buffer_copy(layer)
        setattr(changed, field, value)
        assert call(changed) == code
        assert lib.dflash_encoder_layer_workspace_bytes(byref(changed), 2, 32) == 0
    torch.cuda.synchronize()
