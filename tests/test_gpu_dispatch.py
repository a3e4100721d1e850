"""Which GEMM runs a projection: the hand-written one (``dflash_linear_fwd``,
``dflash_output_block_fwd``) or the library's, seen by recording the calls."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture
def ran(monkeypatch):
    """(op, rows, N, K) of every projection: "hip" or "library"."""

    from torch.nn import functional as F

    from disentangled_flash import layers

    calls = []

    def record(kind, function):
        def call(x, weight, *args):
            calls.append((kind, x.numel() // x.shape[-1], *weight.shape))
            return function(x, weight, *args)
        return call

    monkeypatch.setattr(layers, "linear_epilogue", record("hip", layers.linear_epilogue))
    monkeypatch.setattr(layers, "linear_add_layernorm", record("hip", layers.linear_add_layernorm))
    monkeypatch.setattr(F, "linear", record("library", F.linear))
    return calls


def _blocks(hidden, inner, dtype):
    from transformers import DebertaV2Config
    from transformers.models.deberta_v2.modeling_deberta_v2 import (
        DebertaV2Intermediate,
        DebertaV2Output,
        DebertaV2SelfOutput,
    )

    cfg = DebertaV2Config(hidden_size=hidden, intermediate_size=inner, hidden_act="gelu",
                          hidden_dropout_prob=0.0, layer_norm_eps=1e-7)
    return [m(cfg).to("cuda", dtype).eval()
            for m in (DebertaV2SelfOutput, DebertaV2Intermediate, DebertaV2Output)]


def _run(blocks, rows, hidden, inner, dtype):
    from disentangled_flash.layers import intermediate_block, output_block

    x = torch.zeros(1, rows, hidden, device="cuda", dtype=dtype)
    wide = torch.zeros(1, rows, inner, device="cuda", dtype=dtype)
    with torch.inference_mode():
        output_block(blocks[0], x, x)
        intermediate_block(blocks[1], x)
        output_block(blocks[2], wide, x)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hidden", [256, 768])
def test_projections_by_rows(ran, dtype, hidden):
    inner = 4 * hidden
    blocks = _blocks(hidden, inner, dtype)
    for rows in (1, 512, 4096, 8191, 8192, 16384):
        ran.clear()
        _run(blocks, rows, hidden, inner, dtype)
        last = "library" if rows >= 8192 else "hip"
        assert ran == [("hip", rows, hidden, hidden), ("hip", rows, inner, hidden),
                       (last, rows, hidden, inner)]
    # The same while a HIP graph is captured.
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    ran.clear()
    with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
        _run(blocks, 512, hidden, inner, dtype)
    torch.cuda.current_stream().wait_stream(side)
    assert [kind for kind, *_ in ran] == ["hip"] * 3


def test_what_does_not_fit_runs_in_the_library(ran, monkeypatch):
    from disentangled_flash import layers

    _run(_blocks(256, 1024, torch.float32), 64, 256, 1024, torch.float32)
    _run(_blocks(320, 1280, torch.float16), 64, 320, 1280, torch.float16)
    monkeypatch.setattr(layers, "USE_HIP_GEMM", False)
    _run(_blocks(256, 1024, torch.float16), 64, 256, 1024, torch.float16)
    # 320 columns are no multiple of 128 or 192; 1280 are.
    assert [kind for kind, _, n, _ in ran if n != 1280] == ["library"] * 8
    assert [kind for kind, _, n, _ in ran if n == 1280] == ["hip"]
