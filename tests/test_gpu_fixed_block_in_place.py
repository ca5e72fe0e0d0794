"""Fixed-block dispatch on tensors the kernels read in place, against the same call on contiguous copies.

The copies take the route every call took before (normalised to contiguous [BH,T,D]); both ways run one kernel on the
same rows, so the results are equal bit for bit, shape and strides included.
"""
from __future__ import annotations

import pytest
import torch

from rdna35_block_attention import dispatch, fixed_block_attention

B, H, T, D = 2, 3, 150, 64


def _bhtd(form, gen, dtype):
    def one():
        if form == "contiguous":
            return torch.randn((B, H, T, D), generator=gen).to(dtype)
        if form == "transposed":          # [B,T,H,D] storage
            return torch.randn((B, T, H, D), generator=gen).to(dtype).transpose(1, 2)
        if form == "sliced_heads":
            return torch.randn((B, 2 * H, T, D), generator=gen).to(dtype)[:, ::2]
        if form == "odd_rows":            # rows of D + 1 elements: not 16-byte aligned
            return torch.randn((B, H, T, D + 1), generator=gen).to(dtype)[..., :D]
        return torch.randn((B, H, D, T), generator=gen).to(dtype).transpose(2, 3)  # "strided_dims"
    return one(), one(), one()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("form", ["contiguous", "transposed", "sliced_heads", "odd_rows", "strided_dims"])
@pytest.mark.parametrize("mask_kind", [None, "2d", "4d"])
def test_bhtd_views_match_contiguous_copies(monkeypatch, dtype, form, mask_kind):
    gen = torch.Generator().manual_seed(11)
    q, k, v = (t.cuda() for t in _bhtd(form, gen, dtype))
    q, k, v = (t if form == "contiguous" else _like(t, form) for t in (q, k, v))
    mask = {None: None, "2d": torch.rand((T, T), generator=gen) < 0.8,
            "4d": torch.randn((B, 1, T, T), generator=gen)}[mask_kind]
    mask = None if mask is None else mask.cuda()
    out = fixed_block_attention(q, k, v, layout="bhtd", causal=True, mask=mask)
    monkeypatch.setattr(dispatch, "_in_place_views", lambda *args: None)
    before = fixed_block_attention(q, k, v, layout="bhtd", causal=True, mask=mask)
    assert out.shape == before.shape and out.stride() == before.stride()
    assert torch.equal(torch.nan_to_num(out, nan=7.0), torch.nan_to_num(before, nan=7.0))


def _like(t, form):
    """t on the GPU with the strides its form names (a device copy of a view is contiguous)."""
    if form == "transposed":
        return t.transpose(1, 2).contiguous().transpose(1, 2)
    if form == "sliced_heads":
        return torch.stack((t, t), dim=2).flatten(1, 2)[:, ::2]
    if form == "odd_rows":
        return torch.nn.functional.pad(t, (0, 1))[..., :D]
    return t.transpose(2, 3).contiguous().transpose(2, 3)


@pytest.mark.gpu
@pytest.mark.parametrize("fused", [False, True])
def test_bthd_layout_matches_contiguous_copies(monkeypatch, fused):
    """[B,T,H*D] calls, also as a third of one fused projection, store [B,T,H*D] directly."""
    gen = torch.Generator().manual_seed(12)
    x = torch.randn((B, T, 3 * H * D), generator=gen).to(torch.float16).cuda()
    q, k, v = x.chunk(3, dim=2)
    if not fused:
        q, k, v = (t.contiguous() for t in (q, k, v))
    out, info = fixed_block_attention(q, k, v, layout="bthd", heads=H, return_diagnostics=True)
    monkeypatch.setattr(dispatch, "_in_place_views", lambda *args: None)
    before, info_before = fixed_block_attention(q, k, v, layout="bthd", heads=H, return_diagnostics=True)
    assert out.stride() == before.stride() and torch.equal(out, before) and info == info_before


def test_rows_readable_needs_unit_stride_and_aligned_rows():
    x = torch.zeros((B, H, T, D), dtype=torch.bfloat16)
    assert dispatch._rows_readable(x) and dispatch._rows_readable(x.transpose(0, 1))
    assert not dispatch._rows_readable(x.transpose(2, 3))
    assert not dispatch._rows_readable(torch.zeros((B, H, T, D + 4), dtype=torch.bfloat16)[..., :D])
    assert dispatch._rows_readable(torch.zeros((B, H, T, D + 4), dtype=torch.float32)[..., :D])
    assert not dispatch._rows_readable(torch.zeros(B * H * T * D + 1, dtype=torch.bfloat16)[1:].view(B, H, T, D))
    assert dispatch._in_place_views(x, x, x, "bhtd", None) is None  # CPU tensors take the eager route


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["bhtd", "bthd"])
def test_strided_inputs_that_require_grad_run_the_kernel_with_grad_mode_off(layout):
    """Their contiguous copies do not require grad; with grad mode on the call is the eager path's."""
    gen = torch.Generator().manual_seed(13)
    x = torch.randn((B, T, 3 * H * D), generator=gen).to(torch.bfloat16).cuda().requires_grad_()
    plain = x.detach()

    def call(t):
        q, k, v = t.chunk(3, dim=2)
        if layout == "bhtd":
            q, k, v = (p.view(B, T, H, D).transpose(1, 2) for p in (q, k, v))
        return fixed_block_attention(q, k, v, layout=layout, heads=H, return_diagnostics=True)

    for off in (torch.no_grad, torch.inference_mode):
        with off():
            out, info = call(x)
        assert info["backend"] == "hip" and torch.equal(out, call(plain)[0])
    _, info = call(x)
    assert info["fallback_reason"] == "requires_grad_uses_reference"


def test_tensors_wrapped_by_a_transform_are_not_readable():
    x = torch.zeros((2, B, H, T, D))
    assert torch.func.vmap(lambda t: t.sum() * dispatch._rows_readable(t))(x).tolist() == [0.0, 0.0]


@pytest.mark.gpu
def test_vmap_of_a_call_the_kernel_does_not_take():
    """Head dim 48 falls back to the eager path, under vmap as outside it."""
    gen = torch.Generator().manual_seed(14)
    q, k, v = (torch.randn((2, B, H, T, 48), generator=gen).cuda() for _ in range(3))
    out = torch.func.vmap(lambda *qkv: fixed_block_attention(*qkv, layout="bhtd"))(q, k, v)
    for i in range(2):
        expected = fixed_block_attention(q[i], k[i], v[i], layout="bhtd")
        torch.testing.assert_close(out[i], expected, atol=1e-5, rtol=1e-5)  # fp32 products in another batching


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["bhtd", "bthd"])
def test_a_subclassed_mask_gives_its_type_to_the_result(layout):
    class Mask(torch.Tensor):
        pass

    gen = torch.Generator().manual_seed(15)
    shape = (B, H, T, D) if layout == "bhtd" else (B, T, H * D)
    q, k, v = (torch.randn(shape, generator=gen).cuda() for _ in range(3))
    mask = (torch.rand((T, T), generator=gen) < 0.8).cuda()
    out = fixed_block_attention(q, k, v, layout=layout, heads=H, mask=mask.as_subclass(Mask))
    assert type(out) is Mask
    assert torch.equal(out.as_subclass(torch.Tensor), fixed_block_attention(q, k, v, layout=layout, heads=H, mask=mask))
