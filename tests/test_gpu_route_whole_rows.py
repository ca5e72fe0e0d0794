"""Routing scores at head dims 64 and 128, whose rows the kernel holds and loads whole (at 128 above 64 blocks), on the
MI355X.

The same centroids with 16 zero dims appended take the general loop over the row, which forms the same products in the
same order and adds zeros, so scores and selections must be equal bit for bit.  Against a float64 product the fp32 sums
of D terms are off by at most D * 2^-24 times the sum of their magnitudes (times the scale, rounded once more).
"""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("round_bf16", [False, True])
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("blocks", [1, 15, 16, 17, 63, 64, 65, 81, 129, 256, 257, 513, 1024])
def test_whole_row_scores_equal_the_general_loop(blocks, head_dim, round_bf16):
    import mi355x_pisa

    gen = torch.Generator().manual_seed(blocks + head_dim)
    qc, kc = (torch.randn((2, blocks, head_dim), generator=gen) for _ in range(2))
    k, scale = max(1, blocks // 5), head_dim ** -0.5
    scores, idx = mi355x_pisa.route_topk(qc.cuda(), kc.cuda(), None, k, scale, None, round_bf16=round_bf16)
    wide = [torch.nn.functional.pad(t, (0, 16)).cuda() for t in (qc, kc)]
    general, general_idx = mi355x_pisa.route_topk(*wide, None, k, scale, None, round_bf16=round_bf16)
    assert torch.equal(scores, general)
    assert torch.equal(idx, general_idx)
    a, b = ((t.bfloat16() if round_bf16 else t).double() for t in (qc, kc))
    bound = (head_dim + 1) * 2.0 ** -24 * scale * (a.abs() @ b.abs().transpose(1, 2).contiguous())
    assert bool(((scores.cpu().double() - scale * (a @ b.transpose(1, 2).contiguous())).abs() <= bound).all())
