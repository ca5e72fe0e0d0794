"""The attention calls a user of this package makes, as measurable cases.

A case is one call of a public entry point on inputs that are already on the
GPU, the way the ComfyUI overrides and the Python API issue it once per layer
and sampling step:

* ``fixed``   - rdna35_block_attention.fixed_block_attention: 64-token
  block-diagonal attention, fp32/bf16/fp16, causal and masked;
* ``dense``   - mi355x_pisa.dense_attention: exact self- and cross-attention,
  bf16/fp16, any head dim, also on strided views of one fused QKV projection;
* ``pisa``    - rdna35_block_attention.pisa_attention on flat [BH,T,128];
* ``spatial`` - mi355x_pisa.forward_spatial_bhtd, the 96x96-token image call;
* ``video``   - mi355x_pisa.generic_forward on a (frames, height, width) grid.

Everything is forward-only: the package has no backward.
"""
from __future__ import annotations

import math
import pathlib
import sys

import torch

_PACKAGE = pathlib.Path(__file__).resolve().parents[1] / "comfyui-rdna35-attention_amd"
if str(_PACKAGE) not in sys.path:
    sys.path.insert(0, str(_PACKAGE))

BLOCK = 64
SIDE = 96  # token grid of the spatial call
_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


# ------------------------------------------------------------------ cases
def _fixed(dtype, batch, heads, tokens, dim, causal=False, mask="none", **name):
    return {**name, "kind": "fixed", "dtype": dtype, "batch": batch, "heads": heads, "tokens": tokens, "dim": dim,
            "causal": causal, "mask": mask}


def _dense(dtype, batch, heads, tokens, kv_tokens, dim, fused=False, **name):
    return {**name, "kind": "dense", "dtype": dtype, "batch": batch, "heads": heads, "tokens": tokens,
            "kv_tokens": kv_tokens, "dim": dim, "fused_qkv": fused}


def _pisa(dtype, heads, tokens, budget, **name):
    return {**name, "kind": "pisa", "dtype": dtype, "batch": 1, "heads": heads, "tokens": tokens, "dim": 128,
            "exact": max(1, min(_blocks(tokens), math.ceil(budget * _blocks(tokens)))), "first_order": True}


def _spatial(batch, heads, **name):
    return {**name, "kind": "spatial", "dtype": "bf16", "batch": batch, "heads": heads, "tokens": SIDE * SIDE,
            "dim": 128, "exact": 23, "first_order": True, "frames": 1, "height": SIDE, "width": SIDE}


def _video(dtype, heads, frames, height, width, dim, exact, **name):
    # the override asks for the first-order term at head dim 128 in bf16 only
    return {**name, "kind": "video", "dtype": dtype, "batch": 1, "heads": heads, "tokens": frames * height * width,
            "dim": dim, "exact": exact, "first_order": dim == 128 and dtype == "bf16", "frames": frames,
            "height": height, "width": width}


def _blocks(tokens):
    return (tokens + BLOCK - 1) // BLOCK


def listed():
    return [
        # a small block-diagonal layer: launch and host time
        _fixed("bf16", 1, 8, 256, 64, name="fixed-small"),
        # the default precision of the block-diagonal entry point at an ordinary size
        _fixed("fp32", 1, 8, 4096, 64, name="fixed-fp32"),
        # an additive [T,T] mask with closed entries over a ragged length, shared by the heads
        _fixed("bf16", 2, 16, 4000, 64, mask="add", name="fixed-masked"),
        # the largest block-diagonal layer: an image of 96x96 tokens, two guidance halves
        _fixed("bf16", 2, 16, 9216, 128, name="fixed-large"),
        # a low-resolution stage: few heads and an odd length
        _dense("fp16", 1, 8, 1000, 1000, 64, name="dense-small"),
        # self-attention of a mid-resolution stage at head dim 64
        _dense("fp16", 2, 10, 4096, 4096, 64, name="dense-d64"),
        # image tokens against a 512-token text context
        _dense("bf16", 2, 16, 9216, 512, 128, name="dense-cross"),
        # exact attention read in place from a fused QKV projection
        _dense("bf16", 1, 56, 9170, 9170, 128, fused=True, name="dense-fused-qkv"),
        # sparse attention of a ragged sequence at the API's default budget of a quarter
        _pisa("bf16", 24, 4001, 0.25, name="pisa-ragged"),
        # the 96x96 image call with both guidance halves in one batch
        _spatial(2, 16, name="spatial-image"),
        # video tokens at head dim 64, half precision, a quarter of the blocks exact
        _video("fp16", 32, 16, 32, 32, 64, 64, name="video-d64"),
        # a long video: 32768 tokens, about 16 % of the blocks exact
        _video("bf16", 40, 16, 32, 64, 128, 80, name="video-long"),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """One more call of the ranges above, with at most about the work of the largest of its kind."""
    case = _draw(rng)
    most = {"dense": 2.4e12 if case["dim"] == 128 else 1.2e12, "video": 3.6e12}.get(case["kind"], math.inf)
    flops = work(case)["flops"]
    if flops > most and case["heads"] != 56:
        case["heads"] = max(1, int(case["heads"] * most / flops))
    return case


def _draw(rng):
    kind = rng.choice(("fixed", "fixed", "dense", "dense", "dense", "pisa", "spatial", "video"))
    if kind == "fixed":
        mask = rng.choice(("none", "none", "bool", "add"))
        return _fixed(rng.choice(("bf16", "fp16", "fp32")), rng.randint(1, 2), rng.randint(4, 24),
                      _log_int(rng, 64, 9216 if mask == "none" else 6000), rng.choice((32, 64, 128)),
                      causal=rng.random() < 0.3, mask=mask)
    if kind == "dense":
        if rng.random() < 0.2:
            tokens = _log_int(rng, 4608, 9170)
            return _dense("bf16", 1, 56, tokens, tokens, 128, fused=True)
        tokens = _log_int(rng, 64, 9216)
        kv_tokens = tokens if rng.random() < 0.6 else _log_int(rng, 64, 1024)
        return _dense(rng.choice(("bf16", "fp16")), rng.randint(1, 2), rng.randint(4, 24), tokens, kv_tokens,
                      rng.choice((40, 64, 64, 80, 128, 128, 160)))
    if kind == "pisa":
        return _pisa(rng.choice(("bf16", "bf16", "fp16")), rng.randint(4, 32), _log_int(rng, 1000, 9216),
                     rng.uniform(0.1, 0.5))
    if kind == "spatial":
        return _spatial(rng.randint(1, 2), rng.randint(8, 24))
    dim, dtype = rng.choice(((64, "fp16"), (64, "bf16"), (128, "bf16"), (128, "fp16")))
    frames, height, width = rng.randint(9, 16), 8 * rng.randint(4, 5), 8 * rng.randint(4, 6)
    budget = rng.uniform(0.1, 0.25) if dim == 128 and dtype == "bf16" else 0.25
    return _video(dtype, rng.randint(8, 40), frames, height, width, dim,
                  math.ceil(budget * _blocks(frames * height * width)))


# ------------------------------------------------------------------ inputs
def _smooth(gen, batch, channels, grid):
    """Image or video activations: per channel a unit-variance random field that is smooth over about 8 tokens, plus
    0.3 N(0,1) noise; [batch, tokens, channels] fp32."""
    x = torch.randn((batch, channels, *grid), generator=gen, device="cuda")
    for axis, size in enumerate(grid):
        freq = torch.fft.fftfreq(size, device="cuda")
        gain = torch.exp(-0.5 * (2.0 * math.pi * 8.0 * freq) ** 2)
        spectrum = torch.fft.fft(x, dim=2 + axis) * gain.view([-1 if a == axis else 1 for a in range(len(grid))])
        x = torch.fft.ifft(spectrum, dim=2 + axis).real
    x = x.flatten(2)
    x = (x - x.mean(dim=-1, keepdim=True)) / x.std(dim=-1, keepdim=True).clamp_min(1e-6)
    x = x + 0.3 * torch.randn(x.shape, generator=gen, device="cuda")
    return x.transpose(1, 2)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, dtype = case["kind"], _DTYPES[case["dtype"]]
    batch, heads, tokens, dim = case["batch"], case["heads"], case["tokens"], case["dim"]
    state = {"case": dict(case), "mask": None}
    if kind in ("fixed", "dense"):
        normal = lambda shape: torch.randn(shape, generator=gen, device="cuda").to(dtype)  # noqa: E731
        if kind == "dense" and case["fused_qkv"]:
            fused = normal((batch, tokens, 3, heads, dim))
            state["q"], state["k"], state["v"] = (fused[:, :, i].transpose(1, 2) for i in range(3))
            return state
        kv_tokens = case["kv_tokens"] if kind == "dense" else tokens
        state["q"] = normal((batch, heads, tokens, dim))
        state["k"] = normal((batch, heads, kv_tokens, dim))
        state["v"] = normal((batch, heads, kv_tokens, dim))
        if kind == "fixed" and case["mask"] != "none":
            # a fifth of the entries closed, never a token's own
            closed = torch.rand((tokens, tokens), generator=gen, device="cuda") < 0.2
            closed.fill_diagonal_(False)
            if case["mask"] == "bool":
                state["mask"] = ~closed
            else:
                bias = torch.randn((tokens, tokens), generator=gen, device="cuda").to(dtype)
                state["mask"] = bias.masked_fill_(closed, torch.finfo(dtype).min)
        return state
    grid = (case["frames"], case["height"], case["width"]) if "frames" in case else (tokens,)
    grid = tuple(size for size in grid if size > 1)
    for name in "qkv":
        x = _smooth(gen, batch, heads * dim, grid).to(dtype).reshape(batch, tokens, heads, dim)
        # pisa takes flat [BH,T,D]; the others read [B,T,H,D] storage through a [B,H,T,D] view
        state[name] = x.permute(0, 2, 1, 3)
        if kind == "pisa":
            state[name] = state[name].reshape(batch * heads, tokens, dim).contiguous()
        else:
            state[name] = x.contiguous().permute(0, 2, 1, 3)
    return state


# ------------------------------------------------------------------ the calls
def run(state):
    case, q, k, v = state["case"], state["q"], state["k"], state["v"]
    if case["kind"] == "fixed":
        from rdna35_block_attention import fixed_block_attention

        return fixed_block_attention(q, k, v, layout="bhtd", causal=case["causal"], mask=state["mask"])
    if case["kind"] == "pisa":
        from rdna35_block_attention.pisa_attention import pisa_attention

        return pisa_attention(q, k, v, exact_blocks=case["exact"])
    import mi355x_pisa

    if case["kind"] == "dense":
        return mi355x_pisa.dense_attention(q, k, v, case["dim"] ** -0.5, merged_output=True)
    if case["kind"] == "spatial":
        return mi355x_pisa.forward_spatial_bhtd(q, k, v, case["exact"])
    return mi355x_pisa.generic_forward(q, k, v, case["exact"], case["dim"] ** -0.5, case["first_order"],
                                       token_grid=(case["frames"], case["height"], case["width"]))


# ------------------------------------------------------------------ what a call cannot do without
def work(case):
    heads, tokens, dim = case["batch"] * case["heads"], case["tokens"], case["dim"]
    size = 4 if case["dtype"] == "fp32" else 2
    if case["kind"] == "fixed":
        mask_entry = {"none": 0, "bool": 1, "add": size}[case["mask"]]
        return {"bytes": 4 * heads * tokens * dim * size + tokens * BLOCK * mask_entry,
                "flops": 4 * heads * tokens * BLOCK * dim}
    if case["kind"] == "dense":
        kv_tokens = case["kv_tokens"]
        return {"bytes": 2 * heads * (tokens + kv_tokens) * dim * size, "flops": 4 * heads * tokens * kv_tokens * dim}
    blocks = _blocks(tokens)
    exact, tail = case["exact"], blocks - case["exact"]
    flops = 4 * heads * tokens * dim * (exact * BLOCK + tail)  # exact tiles, centroid tail
    flops += 2 * heads * blocks * blocks * dim  # routing scores
    if case["first_order"]:
        flops += 4 * heads * tokens * dim * dim  # the block covariances and the correction
    return {"bytes": 4 * heads * tokens * dim * size, "flops": flops}


# ------------------------------------------------------------------ results
def tolerance(case):
    # About four times the error measured against exact(): 2.1e-7 in fp32; 2.4e-3 in bf16 and 2.9e-4 in fp16 for exact
    # attention (the rounding of the probabilities and of the output); 2.2e-3 and 2.1e-4 for the sparse calls, whose
    # fp16 bound also leaves room for a query block that takes the other of two key blocks with nearly equal routing
    # scores (its 64 rows move by a few percent, the reason for the wider "max" too).
    if case["kind"] == "fixed":
        return {"rel": {"fp32": 1e-6, "bf16": 1e-2, "fp16": 1.2e-3}[case["dtype"]]}
    if case["kind"] == "dense":
        return {"rel": {"bf16": 1e-2, "fp16": 1.2e-3}[case["dtype"]]}
    return {"rel": {"bf16": 8e-3, "fp16": 2e-3}[case["dtype"]], "max": 0.5}


def _softmax64(scores):
    return torch.softmax(scores, dim=-1)


def exact(case, seed):
    state = prepare(case, seed)
    q, k, v = state["q"], state["k"], state["v"]
    scale = case["dim"] ** -0.5
    if case["kind"] == "fixed":
        return _exact_fixed(q.double(), k.double(), v.double(), scale, case["causal"], state["mask"])
    if case["kind"] == "dense":
        batch, heads, tokens, dim = q.shape
        out = torch.empty((batch, tokens, heads, dim), dtype=torch.float64, device=q.device)
        for b in range(batch):
            for h in range(heads):
                scores = q[b, h].double() @ k[b, h].double().t().contiguous() * scale
                out[b, :, h] = _softmax64(scores) @ v[b, h].double()
        return out.reshape(batch, tokens, heads * dim)
    q4, k4, v4 = (x.unsqueeze(0) if x.ndim == 3 else x for x in (q, k, v))
    order = _block_order(case).to(q.device)
    # routing means: the HYD call (bf16, 128) multiplies bf16 means and adds ln of the covariance norm, the generic
    # one rounds at most the query mean
    hyd = case["kind"] == "spatial" or (case["kind"] == "pisa" and case["dtype"] == "bf16")
    generic_hyd = not hyd and case["kind"] == "video" and case["dim"] == 128 and case["dtype"] == "bf16" \
        and case["tokens"] <= 9216
    out = torch.empty(q4.shape, dtype=torch.float64, device=q.device)
    for b in range(q4.shape[0]):
        for h in range(q4.shape[1]):
            rows = [x[b, h].double()[order] for x in (q4, k4, v4)]
            out[b, h, order] = _exact_sparse(*rows, case["exact"], scale, case["first_order"], hyd, generic_hyd,
                                             q.dtype)
    if case["kind"] == "pisa":
        return out[0]
    out = out.transpose(1, 2).contiguous()  # [B,T,H,D]
    return out.flatten(2) if case["kind"] == "spatial" else out


def _exact_fixed(q, k, v, scale, causal, mask):
    out = torch.empty_like(q)
    for start in range(0, q.shape[2], BLOCK):
        rows = slice(start, min(start + BLOCK, q.shape[2]))
        scores = q[:, :, rows] @ k[:, :, rows].transpose(-1, -2).contiguous() * scale
        if causal:
            n = scores.shape[-1]
            later = torch.ones((n, n), dtype=torch.bool, device=q.device).triu_(1)
            scores = scores.masked_fill(later, -torch.inf)
        if mask is not None and mask.dtype == torch.bool:
            scores = scores.masked_fill(~mask[rows, rows], -torch.inf)
        elif mask is not None:
            scores = scores + mask[rows, rows].double()
        out[:, :, rows] = _softmax64(scores) @ v[:, :, rows]
    return out


def _block_order(case):
    """Raster token of every block-major position: per-frame 8x8 tiles of a token grid, else the sequence itself."""
    if "frames" not in case:
        return torch.arange(case["tokens"])
    frames, height, width = case["frames"], case["height"], case["width"]
    raster = torch.arange(case["tokens"]).reshape(frames, height // 8, 8, width // 8, 8)
    return raster.transpose(2, 3).reshape(-1)


def _exact_sparse(q, k, v, exact_blocks, scale, first_order, hyd, generic_hyd, dtype):
    """One head in block-major order: top-k key blocks of every query block exactly, the others by their centroids and
    the summed key/value covariance."""
    tokens, dim = q.shape
    blocks = _blocks(tokens)
    pad = blocks * BLOCK - tokens
    qb, kb, vb = (torch.nn.functional.pad(x, (0, 0, 0, pad)).reshape(blocks, BLOCK, dim) for x in (q, k, v))
    length = torch.full((blocks,), float(BLOCK), dtype=torch.float64, device=q.device)
    length[-1] = BLOCK - pad
    live = torch.arange(BLOCK, device=q.device)[None, :] < length[:, None]
    q_mean, k_mean, v_mean = (x.sum(dim=1) / length[:, None] for x in (qb, kb, vb))
    centred = (kb - k_mean[:, None, :]) * live[..., None]
    cov = centred.transpose(1, 2).contiguous() @ vb  # [N, D, D]
    if hyd:
        scores = q_mean.to(dtype).double() @ k_mean.to(dtype).double().t().contiguous() * scale
        scores = scores + torch.log(cov.flatten(1).norm(dim=1) + 1e-5)[None, :]
    else:
        scores = (q_mean.to(dtype).double() if generic_hyd else q_mean) @ k_mean.t().contiguous() * scale
    chosen = scores.topk(exact_blocks, dim=-1).indices  # [N, k]
    k_sel, v_sel = (x[chosen].reshape(blocks, -1, dim) for x in (kb, vb))
    s_exact = qb @ k_sel.transpose(1, 2).contiguous() * scale
    s_exact = s_exact.masked_fill(~live[chosen].reshape(blocks, 1, -1), -torch.inf)
    s_tail = qb @ k_mean.t().contiguous() * scale + torch.log(length)
    is_chosen = torch.zeros((blocks, blocks), dtype=torch.bool, device=q.device).scatter_(1, chosen, True)
    s_tail = s_tail.masked_fill(is_chosen[:, None, :], -torch.inf)
    weights = _softmax64(torch.cat((s_exact, s_tail), dim=-1))
    tail = weights[..., s_exact.shape[-1]:]
    out = weights[..., : s_exact.shape[-1]] @ v_sel + tail @ v_mean
    if first_order:
        out = out + (qb @ cov.sum(dim=0)) * (scale / tokens) * tail.sum(dim=-1, keepdim=True)
    return out.reshape(-1, dim)[:tokens]
