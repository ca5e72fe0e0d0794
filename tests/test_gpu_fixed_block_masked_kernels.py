"""Masked fixed-block calls on the matrix-core kernels against the fp32 kernel they ran on before.

16-byte aligned rows take the matrix-core kernels, any other rows the VALU kernel (which stages the block in fp32):
the same call on aligned and on shifted storage compares the two over mask kinds, mask strides, ragged lengths,
head dims, causal masking and values that are not finite.

Both hold scores, probabilities and sums in fp32, so before the output's rounding they differ by the order of at
most 128 products per score (|s| < 16) and 64 per output: (128 * 16 + 64) * 2^-24 max|v| < 1.3e-4 max|v| at worst;
the rounding to 16 bits can then fall on the next value, 2^-7 of it in bf16 and 2^-10 in fp16.
"""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
STEP = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 0.0}


@pytest.fixture(scope="module")
def native():
    import mi355x_pisa

    return mi355x_pisa


def _shifted(x):
    """A copy of x whose rows start one element past a multiple of their width."""
    buf = torch.zeros((*x.shape[:-1], x.shape[-1] + 1), dtype=x.dtype, device=x.device)
    buf[..., 1:] = x
    return buf[..., 1:]


def _mask(kind, shape, gen):
    closed = torch.rand(shape, generator=gen) < 0.3
    if kind == torch.bool:
        return ~closed
    bias = torch.randn(shape, generator=gen).to(kind)
    lowest = torch.where(torch.rand(shape, generator=gen) < 0.5, torch.finfo(kind).min, float("-inf"))
    return torch.where(closed, lowest.to(kind), bias)


def _compare(native, q, k, v, causal, view):
    q, k, v = (t.cuda() for t in (q, k, v))
    out = native.fixed_block_attention(q, k, v, q.shape[-1] ** -0.5, causal, view).float().cpu()
    general = native.fixed_block_attention(*map(_shifted, (q, k, v)), q.shape[-1] ** -0.5, causal, view).float().cpu()
    assert torch.equal(torch.isnan(out), torch.isnan(general))
    inf = torch.isinf(general)
    assert torch.equal(out[inf], general[inf]) and not torch.isinf(out[~inf]).any()
    live = torch.isfinite(general)
    atol = 1.3e-4 * float(v.float()[torch.isfinite(v)].abs().max())
    bad = (out - general).abs() > atol + STEP[q.dtype] * general.abs()
    assert not (bad & live).any(), float((out - general)[bad & live].abs().max())
    return general


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("kind", [torch.bool, torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("head_dim,tokens,causal,form", [
    (64, 256, False, "plain"),     # whole blocks, one aligned load per four entries
    (64, 250, True, "plain"),      # rows of an odd length
    (32, 65, False, "plain"),      # a last block of one token
    (128, 190, False, "per_head"),
    (64, 128, False, "transposed"),  # key stride other than one
    (128, 192, True, "sliced"),    # unit stride, unaligned start
    (32, 1, False, "plain"),
])
def test_masked_calls_match_the_general_kernel(native, dtype, kind, head_dim, tokens, causal, form):
    gen = torch.Generator().manual_seed(head_dim + tokens)
    q, k, v = (torch.randn((2, 3, tokens, head_dim), generator=gen).to(dtype) for _ in range(3))
    if form == "per_head":
        view = _mask(kind, (2, 3, tokens, tokens), gen).cuda()
    elif form == "transposed":
        view = _mask(kind, (tokens, tokens), gen).cuda().t().expand(2, 3, tokens, tokens)
    elif form == "sliced":
        view = _mask(kind, (tokens, tokens + 5), gen).cuda()[:, 3:3 + tokens].expand(2, 3, tokens, tokens)
    else:
        view = _mask(kind, (tokens, tokens), gen).cuda().expand(2, 3, tokens, tokens)
    _compare(native, q, k, v, causal, view)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_masked_calls_keep_infinities_and_nan_where_they_were(native, dtype):
    gen = torch.Generator().manual_seed(5)
    tokens = 100
    q, k, v = (torch.randn((1, 2, tokens, 64), generator=gen).to(dtype) for _ in range(3))
    v[0, 0, 10, 3] = float("inf")
    v[0, 0, 99, 5] = float("-inf")  # the last row of a ragged block
    v[0, 1, 20, 7] = float("nan")
    k[0, 1, 70, 0] = float("inf")
    mask = torch.zeros((tokens, tokens))
    mask[12, :64] = float("-inf")
    mask[13, 4] = float("inf")
    mask[14, 6] = float("nan")
    mask[80:90, 99] = float("-inf")
    general = _compare(native, q, k, v, False, mask.cuda().expand(1, 2, tokens, tokens))
    assert torch.isinf(general).any() and torch.isnan(general).any() and torch.isfinite(general).any()
