"""What a user hangs on an encoder's modules after it was prepared is honoured: hooks and a
replaced activation on an intermediate, on few rows (one library call a layer), on many
(op by op) and in captures."""

from __future__ import annotations

import pytest
import torch
from torch.nn.modules import module as torch_module

from test_gpu_module import _encoder_inputs, _encoder_model
from test_gpu_operands import BATCHES, LENGTH, _captured, _encoder, _forward

pytestmark = pytest.mark.gpu


def _inputs(batch):
    hidden, mask = _encoder_inputs(batch, LENGTH, 256, seed=batch)
    return hidden.to("cuda", torch.float16), mask.cuda()


@pytest.mark.parametrize("where", ["", "dense", "intermediate_act_fn", "all modules"])
@pytest.mark.parametrize("pre", [False, True])
def test_hooks_on_an_intermediate_fire(where, pre):
    encoder = _encoder()
    intermediate = encoder.layer[1].intermediate
    target = intermediate.get_submodule(where if where != "all modules" else "")
    calls = []

    def hook(module, *args):
        if module is target:
            calls.append(1)

    if where == "all modules":
        register = torch_module.register_module_forward_pre_hook if pre \
            else torch_module.register_module_forward_hook
    else:
        register = target.register_forward_pre_hook if pre else target.register_forward_hook
    handle = register(hook)
    try:
        for batch in BATCHES:
            calls.clear()
            _forward(encoder, *_inputs(batch))
            assert len(calls) == 1, batch
        calls.clear()
        _captured(encoder, BATCHES[0], *_inputs(BATCHES[0]))
        assert calls
    finally:
        handle.remove()
    calls.clear()
    _forward(encoder, *_inputs(BATCHES[0]))
    assert not calls


@pytest.mark.parametrize("batch", BATCHES)
@pytest.mark.parametrize("change", ["activation", "forward"])
def test_replaced_activation_and_forward(batch, change):
    encoder = _encoder()
    inputs = _inputs(batch)
    before = _forward(encoder, *inputs)
    intermediate = encoder.layer[1].intermediate
    dense = intermediate.dense
    if change == "activation":
        intermediate.intermediate_act_fn = torch.nn.ReLU()
    else:
        intermediate.forward = lambda x: torch.relu(dense(x))
    got = _forward(encoder, *inputs)
    encoder.layer[1].intermediate.__dict__.pop("forward", None)
    # The same by a hook that replaces the result.
    intermediate.register_forward_hook(lambda m, args, out: torch.relu(dense(*args)))
    assert torch.equal(got, _forward(encoder, *inputs))
    assert not torch.equal(got, before)


@pytest.mark.parametrize("name", ["forward_prepared", "_fused_projection"])
def test_overridden_attention_is_called(name):
    encoder = _encoder()
    attention = encoder.layer[0].attention.self
    inputs = _inputs(BATCHES[0])
    want = _forward(encoder, *inputs)
    original = getattr(attention, name)
    calls = []
    setattr(attention, name, lambda *a, **k: calls.append(1) or original(*a, **k))
    assert torch.equal(_forward(encoder, *inputs), want)
    assert calls == [1]
    delattr(attention, name)

    class Counted(type(attention)):
        pass

    setattr(Counted, name, lambda self, *a: calls.append(2) or getattr(type(self).__mro__[1], name)(self, *a))
    attention.__class__ = Counted
    assert torch.equal(_forward(encoder, *inputs), want)
    assert calls == [1, 2]
