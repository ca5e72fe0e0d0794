"""The packing pass that also forms the block means (generic PISA off head dim 128) on the MI355X.

The routing scores are scale * q_bar . k_bar, and with no exact block the output is the softmax over the packed
centroids alone, so the two check the fp32 means and the packed tables at every padded width and on short blocks.
The scores' tolerance: a mean of 64 values below 6 in magnitude is off by at most 64 * 2^-24 * 6, a product of two
such means over D <= 256 dims by D * 2 * 6 * that times the scale, far below the 1e-3 allowed here.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import assert_close, np32, spatial_to_packed
from oracle import pisa as opisa

pytestmark = pytest.mark.gpu
TOL = {torch.float16: 2e-2, torch.bfloat16: 5e-2}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("head_dim", [8, 40, 64, 96, 104, 160, 192, 256])
@pytest.mark.parametrize("tokens,grid", [(65, None), (190, None), (4160, None), (384, (1, 16, 24))])
def test_pack_means_match_float64_means(dtype, head_dim, tokens, grid):
    import mi355x_pisa

    gen = torch.Generator().manual_seed(head_dim + tokens)
    q, k, v = (torch.randn((1, 2, tokens, head_dim), generator=gen).to(dtype) + 0.5 for _ in range(3))
    scale = head_dim ** -0.5
    out, scores, _ = mi355x_pisa.forward_with_routing(q.cuda(), k.cuda(), v.cuda(), 0, scale, mode="generic",
                                                      first_order=False, token_grid=grid)
    packed = [spatial_to_packed(t, *grid) if grid else np32(t).reshape(2, tokens, head_dim) for t in (q, k, v)]
    blocks = (tokens + 63) // 64
    lengths = np.array([min(64, tokens - 64 * b) for b in range(blocks)])
    means = [np.stack([x[:, 64 * b:64 * b + n].astype(np.float64).mean(axis=1) for b, n in enumerate(lengths)], axis=1)
             for x in packed]
    expected = np.einsum("hid,hjd->hij", means[0], means[1]) * scale
    assert_close(np32(scores), expected, 1e-3, 1e-4, f"scores D={head_dim}")
    name = "bf16" if dtype == torch.bfloat16 else "f16"
    ref = opisa.generic_forward(*packed, 0, scale, first_order=False, dtype=name)
    got = spatial_to_packed(out, *grid) if grid else np32(out).reshape(2, tokens, head_dim)
    assert_close(got, ref, TOL[dtype], TOL[dtype], f"centroids D={head_dim}")
