"""Attention where the longest sequences run first: one workgroup per CU, more than one round.

The order only moves work between workgroups, so every row is checked: batches of less than,
exactly and more than the 16 sequences ordered together, groups that do and do not divide by
the 8 XCDs, one-token sequences, lengths past 512, and masks that are right-padded, all kept,
all padded or have holes.  Reference and bounds are those of ``test_gpu_attention``.
"""

from __future__ import annotations

import pytest
import torch

from test_gpu_attention import _check, _inputs, _run_rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pattern", ["right", "none", "all", "holes"])
@pytest.mark.parametrize("batch,heads,length", [(2, 43, 300), (16, 6, 300), (17, 16, 1),
                                                (33, 3, 300), (8, 11, 520)])
@pytest.mark.parametrize("dim,dtype", [(64, torch.float32), (32, torch.float32),
                                       (128, torch.float16), (128, torch.bfloat16)])
def test_every_sequence_runs_once(batch, heads, length, dim, dtype, pattern):
    args = _inputs(batch, heads, length, dim, dtype, pattern, seed=batch + length)
    for has_c2p, has_p2c in ((True, True), (False, True)):
        out = _run_rel(*args, has_c2p, has_p2c)
        _check(out, *args, has_c2p, has_p2c, f"{batch}x{heads}x{length} {pattern}")
