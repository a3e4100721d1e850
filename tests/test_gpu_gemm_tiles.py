"""The GEMM's tile configurations at the sizes where they can go wrong.

Rows around the tile's, K of less than one slab, of half slabs (K = 32 mod 64) and of
fewer slabs than the LDS ring holds, the narrowest N of each configuration, and the
automatic choice.  Reference and bound are those of ``test_gpu_gemm`` (float64 matmul with the dtype's
roundings; two units in the last place plus the fp32 accumulation error).
"""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from test_gpu_gemm import _check, _inputs, _reference, _run

pytestmark = pytest.mark.gpu

# configuration: rows and columns of its tile
TILES = {1: (128, 192), 2: (128, 128), 3: (256, 192), 4: (64, 128), 5: (64, 64), 6: (256, 256),
         7: (128, 192), 8: (128, 128), 9: (128, 64), 10: (64, 64), 11: (32, 64), 0: (256, 64)}


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("config", TILES)
def test_tile_edges(dtype, config):
    rows, columns = TILES[config]
    for epilogue in (0, 1, 2):
        for m in (1, rows - 1, rows + 1, 2 * rows + 17):
            for k in (32, 64, 96, 480, 1056):
                n = columns * (1 if k < 480 else 3)
                x, w, b, r = _inputs(m, k, n, dtype, seed=m + k + n)
                ref, lin, acc = _reference(x, w, b, r, epilogue, dtype)
                code, y = _run(x, w, b, r if epilogue == 2 else None, epilogue, config)
                assert code == 0
                _, excess = _check(y, ref, lin, acc, dtype, epilogue)
                assert excess <= 0, (config, epilogue, m, n, k, excess)


@pytest.mark.parametrize("config", TILES)
def test_columns_must_fit(config):
    x, w, b, _ = _inputs(64, 64, 320, torch.float16, 3)
    code, _ = _run(x, w, b, None, 0, config)
    assert code == (0 if config == 0 or 320 % TILES[config][1] == 0 else -2)
    assert _run(x, w, b, None, 0, 12)[0] == -2


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_gelu_over_its_whole_range(dtype):
    """Bias only (x = 0): every finite input, the infinities and NaN."""

    bits = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dtype).to("cuda")
    x = torch.zeros(1, 32, device="cuda", dtype=dtype)
    w = torch.zeros(65536, 32, device="cuda", dtype=dtype)
    code, y = _run(x, w, bits, None, 1)
    assert code == 0
    ref = F.gelu(bits.double())
    assert torch.equal(torch.isnan(y[0]), torch.isnan(ref))
    finite = torch.isfinite(bits)
    assert torch.equal(y[0][bits == float("inf")], bits[bits == float("inf")])
    # x Phi(x) through erfc, which keeps its relative accuracy in the negative tail.
    x64 = bits[finite].double()
    got, want = y[0][finite].double(), 0.5 * x64 * torch.special.erfc(-x64 * 0.5 ** 0.5)
    # Half a unit in the last place of the result, plus the fp32 evaluation of x Phi(x): the
    # smaller of 4e-7 and 2^-8 relative for its fit (the tail of bf16 reaches 1e-37, where an
    # absolute bound says nothing) and 2^-22 relative for its roundings; past x = -12.9
    # Phi is below the normal fp32 numbers, 13 * 2^-126 of the result at most.
    mantissa = 10 if dtype == torch.float16 else 7
    step = torch.exp2(torch.floor(torch.log2(want.abs().clamp_min(torch.finfo(dtype).tiny))) - mantissa)
    fit = (want.abs() * 2.0 ** -8).clamp_max(4e-7)
    bound = 0.5 * step + fit + want.abs() * 2.0 ** -22 + 13 * 2.0 ** -126
    assert bool(((got - want).abs() <= bound).all())


def test_rows_past_32_bit_offsets():
    """K so long that a tile's rows leave the 32-bit offsets of a buffer resource."""

    k = (1 << 23) + 32
    gen = torch.Generator(device="cuda").manual_seed(2)
    x = torch.randn(3, k, generator=gen, device="cuda").half()
    w = torch.randn(64, k, generator=gen, device="cuda").half()
    w *= k ** -0.5
    b = torch.randn(64, generator=gen, device="cuda").half()
    r = torch.randn(3, 64, generator=gen, device="cuda").half()
    ref, lin, acc = _reference(x, w, b, r, 2, torch.float16)
    for config in (3, 12):  # columns that do not divide N, no configuration
        assert _run(x, w, b, r, 2, config)[0] == -2
    for config in (0, 10, 11):
        code, y = _run(x, w, b, r, 2, config)
        assert code == 0
        # fp32 accumulation over 2^18 MFMA steps one after the other: half a unit in the
        # last place of the running sum (O(1)) each, 2^-24 sqrt(2^18) at random, ten
        # times that allowed.
        _, excess = _check(y, ref, lin, acc + 10 * 2.0 ** -15, torch.float16, 2)
        assert excess <= 0, (config, excess)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("config", [0, 2, 6, 10])
def test_equal_rows(dtype, config):
    """A row's fp32 sums run in an order that depends on its tile: equal rows agree to the
    bound of any order (half a unit of the type each, and the fp32 sums), repeated calls to
    the bit."""

    m, k, n = 2048, 1536, 256
    x, w, b, r = _inputs(1, k, n, dtype, seed=11)
    x, r = x.expand(m, k).contiguous(), r.expand(m, n).contiguous()
    ref, lin, acc = _reference(x, w, b, r, 0, dtype)
    first = None
    for _ in range(3):
        code, y = _run(x, w, b, None, 0, config)
        assert code == 0
        assert first is None or torch.equal(y, first)
        first = y
    _, excess = _check(first, ref, lin, acc, dtype, 0)
    assert excess <= 0


@pytest.mark.parametrize("epilogue", [0, 1])
@pytest.mark.parametrize("m", [8191, 8200])
def test_outputs_around_64_mib(m, epilogue):
    """Outputs below and above the size where plain ones are no longer written through the L2."""

    x, w, b, r = _inputs(m, 96, 4096, torch.bfloat16, seed=m)
    ref, lin, acc = _reference(x, w, b, r, epilogue, torch.bfloat16)
    code, y = _run(x, w, b, None, epilogue)
    assert code == 0
    _, excess = _check(y, ref, lin, acc, torch.bfloat16, epilogue)
    assert excess <= 0
