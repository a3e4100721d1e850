"""``dflash_output_block_fwd``: projection + residual + LayerNorm, with K split for few rows.

Against a float64 evaluation with the dtype's roundings in place.  The projection may
land one rounding step off (its fp32 sums run in another order, more so when K is
split), which moves the rounded sum by at most one step of each: that difference times
gamma / sigma, plus the bound of the fused LayerNorm itself (``test_gpu_layers``).
"""

from __future__ import annotations

import pytest
import torch

from test_gpu_gemm import _inputs, _ulp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m", [1, 16, 33, 64, 200, 513, 1100])
def test_output_block(dtype, m):
    from disentangled_flash import _lib
    from disentangled_flash.layers import linear_add_layernorm

    lib = _lib.load()
    split = 0
    for n, k in ((768, 768), (768, 3072), (1024, 4096), (1536, 6144), (64, 2080), (4096, 1056),
                 (320, 512)):
        x, w, b, r = _inputs(m, k, n, dtype, seed=m + n + k)
        gen = torch.Generator().manual_seed(n)
        gamma = (1 + 0.1 * torch.randn(n, generator=gen)).to("cuda", dtype)
        beta = (0.1 * torch.randn(n, generator=gen)).to("cuda", dtype)
        lin = (x.double() @ w.double().t() + b.double()).to(dtype)
        s = (lin.double() + r.double()).to(dtype)
        mean = s.double().mean(-1, keepdim=True)
        rstd = (s.double().var(-1, unbiased=False, keepdim=True) + 1e-7).rsqrt()
        ref = (s.double() - mean) * rstd * gamma.double() + beta.double()
        acc = (x.double().abs() @ w.double().abs().t() + b.double().abs()) * 2.0 ** -20
        moved = (_ulp(lin.double(), dtype) + _ulp(s.double(), dtype) + acc) * rstd \
            * gamma.double().abs()
        rel, absolute = (2.0 ** -10, 1e-3) if dtype == torch.float16 else (2.0 ** -7, 8e-3)
        tol = moved + moved.mean(-1, keepdim=True) + rel * ref.abs() + absolute
        split += lib.dflash_output_block_workspace_bytes(m, n, k) > 2 * m * n
        for _ in range(2):
            y = linear_add_layernorm(x, w, b, r, gamma, beta, 1e-7)
            excess = ((y.double() - ref).abs() - tol).max().item()
            assert excess <= 0, (m, n, k, excess)
    assert split or m > 512  # few rows: the split form is what ran


def test_output_block_errors():
    from disentangled_flash import _lib
    from disentangled_flash.layers import linear_add_layernorm

    lib = _lib.load()
    x, w, b, r = _inputs(64, 3072, 768, torch.float16, 1)
    g = torch.ones(768, device="cuda", dtype=torch.float16)
    y = torch.empty_like(r)
    size = lib.dflash_output_block_workspace_bytes(64, 768, 3072)
    ws = torch.empty(size, device="cuda", dtype=torch.uint8)
    st = torch.cuda.current_stream().cuda_stream

    def call(res, workspace, bytes_, n=768, k=3072, dtype=0):
        return lib.dflash_output_block_fwd(
            x.data_ptr(), w.data_ptr(), b.data_ptr(), res, g.data_ptr(), g.data_ptr(),
            y.data_ptr(), 64, n, k, 1e-7, dtype, workspace, bytes_, st)

    assert call(r.data_ptr(), ws.data_ptr(), size) == 0
    assert call(None, ws.data_ptr(), size) == -1
    assert call(r.data_ptr(), None, size) == -1
    assert call(r.data_ptr(), ws.data_ptr(), size - 1) == -7
    assert call(r.data_ptr(), ws.data_ptr(), size, dtype=2) == -4
    assert call(r.data_ptr(), ws.data_ptr(), size, n=100) == -2
    with pytest.raises(ValueError):
        linear_add_layernorm(x, w, b, r[:32], g, g, 1e-7)
    empty = linear_add_layernorm(x[:0], w, b, r[:0], g, g, 1e-7)
    assert empty.shape == (0, 768)
