"""The prefill attention (tiq_prefill_attention) at its edges: tiles of 32
queries and blocks of 32 keys (31, 32, 33 of each), one, two and four wavefronts
a tile (by block count, and at 767 / 768 tiles), head counts that leave XCDs
without a pair, a history that starts inside a block, batch-major and
position-major layouts, memory past the last key, and scores far apart.

Bound against float64, derived: a score is a sum of 64 products, its rounding at
most 64 u sum|q k| / 8 <= 8 u |q| |k|; probabilities err by that (an exponent)
and an output by it times max|v|, plus the roundings of S products and sums.
"""
from __future__ import annotations

import pytest
import torch

from gpt2_harness_amd import _lib

pytestmark = pytest.mark.gpu


def _ref(q, k, v, first):
    q, k, v = q.double().contiguous(), k.double().contiguous(), v.double().contiguous()
    T, S = q.shape[-2], k.shape[-2]
    hidden = torch.arange(S, device=q.device)[None, :] > (first + torch.arange(T, device=q.device))[:, None]
    s = (q @ k.transpose(-2, -1).contiguous() / 8.0).masked_fill(hidden, float("-inf"))
    return torch.softmax(s, -1) @ v


def _run(q, k, v, first):
    B, H, T, hd = q.shape
    y = torch.full((B, T, H * hd), float("nan"), device=q.device)
    _lib.check(_lib.lib().tiq_prefill_attention(
        q.data_ptr(), *q.stride()[:3], k.data_ptr(), *k.stride()[:3], v.data_ptr(), *v.stride()[:3], B, H, T, first,
        hd, y.data_ptr(), y.stride(0), hd, y.stride(1), torch.cuda.current_stream().cuda_stream), "attention")
    torch.cuda.synchronize()
    return y


def _check(y, q, k, v, first):
    B, H, T, hd = q.shape
    ref = _ref(q, k, v, first).transpose(1, 2).reshape(B, T, H * hd)
    u = 2.0**-24
    top = float(q.norm(dim=-1).max()) * float(k.norm(dim=-1).max())
    bound = float(v.abs().max()) * u * (2 * 8 * top + k.shape[-2] + 64)
    assert float((y.double() - ref).abs().max()) <= bound


@pytest.mark.parametrize("B,H,T,first", [
    (1, 1, 1, 0), (1, 3, 31, 0), (2, 5, 32, 0), (1, 9, 33, 0), (3, 4, 65, 0), (1, 12, 200, 0),  # 1, 2, 4 wavefronts
    (1, 8, 1, 32), (1, 8, 2, 63), (2, 7, 40, 17), (1, 2, 33, 300),  # a history, block edges inside the tile
    (59, 13, 32, 0), (64, 12, 32, 64),   # 767 and 768 tiles
    (16, 12, 128, 0), (13, 15, 129, 128),  # one wavefront a tile; two from eight blocks
])
@pytest.mark.parametrize("layout", ["cache", "rows"])
def test_prefill_attention_edges(dev, B, H, T, first, layout):
    gen = torch.Generator(device=dev).manual_seed(B + H + T + first)
    S = first + T
    qkv = torch.randn(B, T, 3, H, 64, generator=gen, device=dev)
    q = qkv[:, :, 0].permute(0, 2, 1, 3)
    if layout == "rows":  # (B, S, H, 64) rows
        k, v = (torch.randn(B, S, H, 64, generator=gen, device=dev).permute(0, 2, 1, 3) for _ in range(2))
    else:  # cache buffers, NaN past the last key
        k, v = (torch.full((B, H, S + 37, 64), float("nan"), device=dev) for _ in range(2))
        k[:, :, :S] = torch.randn(B, H, S, 64, generator=gen, device=dev)
        v[:, :, :S] = torch.randn(B, H, S, 64, generator=gen, device=dev)
        k, v = k[:, :, :S], v[:, :, :S]
    _check(_run(q, k, v, first), q, k, v, first)


def test_prefill_attention_far_scores(dev):
    """Scores hundreds apart (the running maximum moves late, whole blocks
    vanish), a query whose every score is equal, and a NaN query."""
    gen = torch.Generator(device=dev).manual_seed(3)
    q, k, v = (torch.randn(1, 2, 160, 64, generator=gen, device=dev) for _ in range(3))
    k[0, 0, 100:] *= 30.0
    q[0, 0, 150] *= 20.0
    q[0, 1, 40] = 0.0
    _check(_run(q, k, v, 0), q, k, v, 0)
    y = _run(q, k, v, 0)
    q[0, 1, 77] = float("nan")
    bad = _run(q, k, v, 0)
    assert bool(bad[0, 77, 64:].isnan().all())
    keep = [t for t in range(160) if t != 77]
    assert torch.equal(bad[0, keep], y[0, keep]) and torch.equal(bad[0, 77, :64], y[0, 77, :64])
