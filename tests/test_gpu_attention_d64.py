"""The split-list attention kernel (head dim 64, and small dense calls up to 128) on the MI355X at the sizes where
its key split and its choice between packed tables and rows in place change.

One to eight waves share a query block and merge their parts of its chunk list; the split follows the number of
query blocks and chunks, so the shapes below reach every split, ragged last blocks, lists shorter than the split
and parts whose every score is masked.

Tolerance of the dense checks: the probabilities and the output are rounded to the storage type (relative 2^-9 in
bf16, 2^-12 in fp16, at most) and an output row is an average of the values with weights that sum to one, so an
element is off by at most (2^-9 + 2^-9) max|v|, twice that bound being allowed.
"""
from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from helpers import assert_close, np32
from oracle import attention as oatt
from oracle import pisa as opisa

pytestmark = pytest.mark.gpu
UNIT = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}
TOL = {torch.bfloat16: 5e-2, torch.float16: 2e-2}


@pytest.fixture(scope="module")
def native():
    import mi355x_pisa

    return mi355x_pisa


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,q_tokens,kv_tokens,head_dim", [
    (1, 1, 1, 64),          # one row, one key
    (2, 65, 77, 64),        # two chunks, the second short
    (3, 130, 1000, 40),     # eight waves, 16 chunks, short last chunk, padded dims
    (40, 300, 1024, 64),    # 200 blocks: four waves
    (20, 1600, 512, 64),    # 500 blocks of 8 chunks: two waves
    (64, 1024, 130, 64),    # 1024 blocks: one wave
    (2, 64, 449, 8),        # eight chunks, the last of one key: four waves
    (3, 130, 1000, 128),    # head dims up to 128 in place: four waves
    (2, 65, 77, 120),       # two chunks
    (40, 500, 500, 104),    # 320 blocks of 8 chunks: two waves
    (64, 1100, 64, 128),    # one chunk: one wave
    (1, 200, 700, 80),      # padded width 96 on the wider kernel
    (5, 6400, 640, 96),     # 500 blocks
    # the shapes above read K and V in place, these from packed tables
    (32, 4096, 512, 96),
    (16, 4096, 1279, 128),
    (1, 7990, 8000, 64),    # 125 blocks of 125 chunks: eight waves
    (2, 6400, 6400, 40),    # 200 blocks: four waves
    (5, 6400, 2500, 64),    # 500 blocks of 40 chunks: two waves
    (25, 2650, 2600, 64),   # 1050 blocks of 41 chunks: four waves, five rounds
    # at most one wave per SIMD: the 512-register kernel
    (16, 4096, 1279, 64),   # 1024 blocks of 20 chunks
    (12, 4090, 2010, 40),   # 768 of 32, padded dims, short last rows and keys
    (14, 2880, 2880, 64),   # 630 of 45
])
def test_dense_splits_match_oracle(native, dtype, heads, q_tokens, kv_tokens, head_dim):
    gen = torch.Generator().manual_seed(heads * 7 + q_tokens + kv_tokens)
    q = torch.randn((1, heads, q_tokens, head_dim), generator=gen).to(dtype)
    k, v = (torch.randn((1, heads, kv_tokens, head_dim), generator=gen).to(dtype) for _ in range(2))
    out = native.dense_attention(q.cuda(), k.cuda(), v.cuda(), 1 / math.sqrt(head_dim))
    rows = slice(None, None, 1 + q_tokens // 200)  # of a long call, some rows of every block
    expected = oatt.dense_attention(np32(q[:, :, rows]), np32(k), np32(v))
    atol = 4 * UNIT[dtype] * float(v.float().abs().max())
    assert_close(np32(out[:, :, rows]), expected, atol, 0.0, f"dense {heads}x{q_tokens}x{kv_tokens} D={head_dim}")


@pytest.mark.parametrize("head_dim,kv_tokens", [(64, 130), (40, 257), (8, 64), (128, 130), (112, 257), (80, 65)])
def test_rows_read_in_place_stay_inside_their_heads(native, head_dim, kv_tokens):
    """Views into one fused [B,T,3,H,D+8] tensor whose other elements are NaN: nothing past a row or past the last
    token reaches the result, an infinite value in the last row stays one column's, and stores end with the row."""
    gen = torch.Generator().manual_seed(head_dim)
    fused = torch.full((2, kv_tokens, 3, 3, head_dim + 8), float("nan"), dtype=torch.bfloat16)
    fused[..., :head_dim] = torch.randn((2, kv_tokens, 3, 3, head_dim), generator=gen).to(torch.bfloat16)
    fused[0, -1, 2, 1, 3] = float("inf")
    fused = fused.cuda()
    q, k, v = (fused[:, :, i, :, :head_dim].transpose(1, 2) for i in range(3))
    out = torch.full((2, 3, kv_tokens, head_dim + 4), 3.0, dtype=torch.bfloat16, device="cuda")  # 8-byte aligned rows
    native._launch_dense(q, k, v, out[..., :head_dim], head_dim ** -0.5)
    expected = oatt.dense_attention(np32(q), np32(k), np32(v))
    assert np.isinf(expected[0, 1, :, 3]).all() and np.isfinite(np.delete(expected, 3, axis=3)).all()
    atol = 4 * UNIT[torch.bfloat16] * 5.0  # |v| < 5
    assert_close(np32(out[..., :head_dim]), expected, atol, 0.0, "in place")
    assert bool((out[..., head_dim:] == 3.0).all())


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("target", ["k", "v"])
def test_output_over_the_keys_or_values(native, head_dim, target):
    """An output stored over K or V: the call then packs them first instead of reading them while it stores.

    4096 query blocks, more than fit the GPU at once: without the packing, late blocks would read stored outputs.
    """
    gen = torch.Generator().manual_seed(9)
    q, rows = (torch.randn((2, 32, 4096, head_dim), generator=gen).to(torch.bfloat16).cuda() for _ in range(2))
    other = torch.randn((2, 32, 64, head_dim), generator=gen).to(torch.bfloat16).cuda()
    k, v = (rows[:, :, :64], other) if target == "k" else (other, rows[:, :, :64])
    expected = native.dense_attention(q, k, v, head_dim ** -0.5)
    native._launch_dense(q, k, v, rows, head_dim ** -0.5)
    assert_close(np32(rows), np32(expected), 4 * UNIT[torch.bfloat16] * 5.0, 0.0, f"out over {target}")


@pytest.mark.parametrize("head_dim", [64, 40, 128, 104, 72])
@pytest.mark.parametrize("kv_tokens", [1, 33, 65, 96, 130, 190])
def test_rows_past_the_last_token_are_never_used(native, kv_tokens, head_dim):
    """Keys and values of a longer buffer whose later rows (and later dims) are NaN."""
    gen = torch.Generator().manual_seed(kv_tokens)
    q = torch.randn((1, 2, 70, head_dim), generator=gen).to(torch.bfloat16)
    k, v = (torch.full((1, 2, kv_tokens + 130, head_dim + 8), float("nan"), dtype=torch.bfloat16) for _ in range(2))
    for t in (k, v):
        t[:, :, :kv_tokens, :head_dim] = torch.randn((1, 2, kv_tokens, head_dim), generator=gen).to(torch.bfloat16)
    k, v = (t.cuda()[:, :, :kv_tokens, :head_dim] for t in (k, v))
    out = native.dense_attention(q.cuda(), k, v, head_dim ** -0.5)
    expected = oatt.dense_attention(np32(q), np32(k), np32(v))
    assert_close(np32(out), expected, 4 * UNIT[torch.bfloat16] * 5.0, 0.0, f"Tk={kv_tokens}")


def test_dense_split_parts_of_very_different_scale(native):
    """Key parts whose maxima lie far apart (and rise along the list) merge without overflow or loss."""
    gen = torch.Generator().manual_seed(3)
    q = torch.randn((1, 2, 64, 64), generator=gen)
    k = torch.randn((1, 2, 512, 64), generator=gen) * torch.linspace(0.0, 12.0, 512)[:, None]
    v = torch.randn((1, 2, 512, 64), generator=gen)
    q, k, v = (t.to(torch.bfloat16) for t in (q, k, v))
    out = native.dense_attention(q.cuda(), k.cuda(), v.cuda(), 1.0)
    expected = oatt.dense_attention(np32(q), np32(k), np32(v), 1.0)
    # scores reach about 400 here: a bf16 product is exact and an fp32 sum of 64 of them is off by up to
    # 64 * 2^-24 * 400, which moves a probability by 0.15 % beside the storage rounding
    atol = (4 * UNIT[torch.bfloat16] + 64 * 2.0 ** -24 * 400) * float(v.float().abs().max())
    assert_close(np32(out), expected, atol, 0.0, "rising scores")


@pytest.mark.parametrize("heads,q_tokens,kv_tokens,head_dim", [
    (1, 70, 832, 64), (1, 70, 512, 128),  # in place: eight waves of one or two chunks, four of two
    (2, 256, 16384, 64),                  # packed: eight waves of 32
])
def test_dense_parts_whose_every_score_is_minus_infinity(native, heads, q_tokens, kv_tokens, head_dim):
    """Keys of minus infinity in a dim where every query is one: their parts weigh nothing in the merge."""
    gen = torch.Generator().manual_seed(kv_tokens + head_dim)
    q = torch.randn((1, heads, q_tokens, head_dim), generator=gen)
    k, v = (torch.randn((1, heads, kv_tokens, head_dim), generator=gen) for _ in range(2))
    q[..., 0] = 1.0
    k[:, :, : kv_tokens // 2, 0] = -math.inf
    k[:, :, kv_tokens // 2 + 100:, 0] = -math.inf
    q, k, v = (t.to(torch.bfloat16) for t in (q, k, v))
    out = native.dense_attention(q.cuda(), k.cuda(), v.cuda(), head_dim ** -0.5)
    live = slice(kv_tokens // 2, kv_tokens // 2 + 100)
    expected = oatt.dense_attention(np32(q), np32(k[:, :, live]), np32(v[:, :, live]))
    assert_close(np32(out), expected, 4 * UNIT[torch.bfloat16] * 5.0, 0.0, f"{kv_tokens} keys, 100 of them live")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,tokens,exact,first_order,scale", [
    (2, 1000, 0, False, 0.125),   # centroids only: one chunk, one wave
    (2, 500, 7, True, 0.125),     # all but one block exact, short last block: four waves
    (1, 4100, 6, True, 0.125),    # two centroid chunks, the second nearly all padding: four waves
    (16, 1024, 4, False, 1e-3),   # a small softmax scale: bias / scale beyond fp16's range
    # the last centroid chunk's second half: only padding (skipped), or one centroid
    (33, 2048, 0, True, 0.125),   # one wave: 32 centroids
    (32, 2103, 3, True, 0.125),   # one wave: 33
    (16, 2043, 9, True, 0.125),   # two waves: 32
    (1, 4140, 20, True, 0.125),   # eight waves: 65, one in the second chunk
])
def test_sparse_splits_match_oracle(native, dtype, heads, tokens, exact, first_order, scale):
    gen = torch.Generator().manual_seed(tokens + exact)
    q, k, v = (torch.randn((1, heads, tokens, 64), generator=gen).to(dtype) for _ in range(3))
    out, scores, idx = native.forward_with_routing(q.cuda(), k.cuda(), v.cuda(), exact, scale, mode="generic",
                                                   first_order=first_order)
    assert (idx.cpu().numpy() == opisa.topk_ascending(scores.cpu().numpy(), exact)).all()
    name = "bf16" if dtype == torch.bfloat16 else "f16"
    ref = opisa.generic_forward(*(np32(t).reshape(heads, tokens, 64) for t in (q, k, v)), exact, scale,
                                first_order=first_order, dtype=name)
    assert_close(np32(out).reshape(heads, tokens, 64), ref, TOL[dtype], TOL[dtype], f"sparse T={tokens}")
