"""Batched decode over int4 codes in operand tiles (tiq_tile_int4,
TIQ_WF_INT4_TILED): a nibble enters the matrix cores as 16 (n - 8), exact in bf16,
and the sums are scaled back by a power of two, so every result equals, bit for
bit, the int8 path's on the same codes held as int8. Then the captured decoder on
an int4 model against the eager one.
"""
from __future__ import annotations

import pytest
import torch

import gpt2_harness_amd as g
from gpt2_harness_amd import _lib

pytestmark = pytest.mark.gpu


def _st():
    return torch.cuda.current_stream().cuda_stream


def _codes(N, K, dev, gen):
    q = torch.randint(-8, 8, (N, K), generator=gen, device=dev).to(torch.int8)
    return q, g.pack_int4(q)


def _tiles(q, packed):
    N, K = q.shape
    L = _lib.lib()
    t8, t4 = torch.empty(N * K, dtype=torch.uint8, device=q.device), torch.empty(N * K // 2, dtype=torch.uint8,
                                                                                 device=q.device)
    _lib.check(L.tiq_tile_int8(q.data_ptr(), N, K, K, t8.data_ptr(), _st()), "tile")
    _lib.check(L.tiq_tile_int4(packed.data_ptr(), N, K, t4.data_ptr(), _st()), "tile")
    return t8, t4


@pytest.mark.parametrize("M", [5, 32, 33, 64])
@pytest.mark.parametrize("K,N", [(32, 32), (768, 2304), (768, 768), (3072, 768), (1600, 6400), (6400, 1600)])
def test_int4_tiles_equal_int8(dev, K, N, M):
    gen = torch.Generator(device=dev).manual_seed(K + N + M)
    q, packed = _codes(N, K, dev, gen)
    x = torch.randn(M, K, generator=gen, device=dev)
    scale = torch.rand(N, generator=gen, device=dev) + 0.5
    bias = torch.randn(N, generator=gen, device=dev)
    ln = [torch.randn(n, generator=gen, device=dev) for n in (K, K, N, N)]
    res = torch.randn(M, N, generator=gen, device=dev)
    L = _lib.lib()
    ws = torch.empty(int(L.tiq_decode_linear_workspace(_lib.WF_INT8_TILED, M, K, N)), dtype=torch.uint8, device=dev)
    assert int(L.tiq_decode_linear_workspace(_lib.WF_INT4_TILED, M, K, N)) == ws.numel()
    outs = []
    for w, wf in zip(_tiles(q, packed), (_lib.WF_INT8_TILED, _lib.WF_INT4_TILED)):
        got = []
        # rows out; LayerNorm in, GELU, planes out; residual and the next LayerNorm's planes
        for kw in ({}, {"ln": True, "act": 1, "planes": True}, {"res": True, "next": True, "planes": True}):
            y = torch.full((M, N), float("nan"), device=dev)
            p = torch.zeros(int(L.tiq_decode_planes_bytes(M, N)), dtype=torch.uint8, device=dev)
            _lib.check(L.tiq_decode_linear(
                x.data_ptr(), K, None, M, K, w.data_ptr(), wf, scale.data_ptr(), bias.data_ptr(), N, y.data_ptr(), N,
                ln[0].data_ptr() if "ln" in kw else None, ln[1].data_ptr() if "ln" in kw else None, 1e-5,
                kw.get("act", 0), res.data_ptr() if "res" in kw else None, N,
                ln[2].data_ptr() if "next" in kw else None, ln[3].data_ptr() if "next" in kw else None, 1e-5,
                p.data_ptr() if "planes" in kw else None, ws.data_ptr(), ws.numel(), _st()), "decode linear")
            got += [y, p]
        outs.append(got)
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    ref = x.double() @ (q.double() * scale.double().unsqueeze(1)).t() + bias.double()
    bound = (x.double().abs() @ (q.double().abs() * scale.double().unsqueeze(1)).t() + bias.double().abs()) * (3 * K + 8) * 2.0**-24
    assert bool(((outs[1][0].double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("B,H", [(5, 12), (33, 4)])
def test_int4_qkv_attention_equals_int8(dev, B, H):
    C, T, pos = 64 * H, 160, 40
    gen = torch.Generator(device=dev).manual_seed(B)
    q, packed = _codes(3 * C, C, dev, gen)
    scale = torch.rand(3 * C, generator=gen, device=dev) * 0.01
    bias = torch.randn(3 * C, generator=gen, device=dev)
    x = torch.randn(B, C, generator=gen, device=dev)
    L = _lib.lib()
    planes = torch.empty(int(L.tiq_decode_planes_bytes(B, C)), dtype=torch.uint8, device=dev)
    t8, t4 = _tiles(q, packed)
    ws = torch.empty(max(int(L.tiq_decode_linear_workspace(_lib.WF_INT8, B, C, 3 * C)),
                         int(L.tiq_decode_qkv_attention_workspace(B, C, 3 * C))), dtype=torch.uint8, device=dev)
    # planes of x itself: an identity-coded linear's planes out
    eye = torch.eye(C, device=dev).to(torch.int8)
    one = torch.ones(C, device=dev)
    _lib.check(L.tiq_decode_linear(x.data_ptr(), C, None, B, C, eye.data_ptr(), _lib.WF_INT8, one.data_ptr(), None, C,
                                   None, 0, None, None, 1e-5, 0, None, 0, None, None, 1e-5, planes.data_ptr(),
                                   ws.data_ptr(), ws.numel(), _st()), "planes")
    p = torch.full((1,), pos, dtype=torch.long, device=dev)
    k0, v0 = (torch.randn(B, H, T, 64, generator=gen, device=dev) for _ in range(2))
    outs = []
    for w, wf in ((t8, _lib.WF_INT8_TILED), (t4, _lib.WF_INT4_TILED)):
        k, v, y = k0.clone(), v0.clone(), torch.empty(B, C, device=dev)
        _lib.check(L.tiq_decode_qkv_attention(planes.data_ptr(), B, C, w.data_ptr(), wf, scale.data_ptr(),
                                              bias.data_ptr(), H, H, 64, k.data_ptr(), v.data_ptr(), T, p.data_ptr(),
                                              y.data_ptr(), C, None, ws.data_ptr(), ws.numel(), _st()), "attention")
        outs.append((k, v, y))
    for a, b in zip(*outs):
        assert torch.equal(a, b)


@pytest.mark.parametrize("batch,bits,granularity", [(5, 4, "per_channel"), (8, 3, "per_tensor"), (40, 4, "per_channel")])
def test_int4_batched_decoder(dev, batch, bits, granularity):
    torch.manual_seed(0)
    cfg = g.GPTConfig(vocab_size=997, n_positions=128, n_layer=2, n_head=4, n_embd=256)
    qm, _ = g.quantize_model(g.GPT(cfg).to(dev).eval(), bits, granularity)
    idx = torch.randint(0, cfg.vocab_size, (batch, 9), device=dev)
    dec = g.FusedDecoder(qm, batch, 40)
    assert dec.chain
    out = dec.run(idx, 20)
    want = g.generate(qm, idx, 20)
    assert torch.equal(out, want)
    with torch.no_grad():
        logits = qm(want[:, :-1])["logits"][:, -1]
    assert torch.allclose(dec.logits, logits, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("bits", [4, 8])
def test_widths_past_the_chain(dev, bits):
    """A block whose c_fc the chain does not take (3072 inputs) keeps one fused
    product a Linear."""
    torch.manual_seed(0)
    cfg = g.GPTConfig(vocab_size=320, n_positions=32, n_layer=1, n_head=48, n_embd=3072)
    qm, _ = g.quantize_model(g.GPT(cfg).to(dev).eval(), bits)
    idx = torch.randint(0, cfg.vocab_size, (6, 4), device=dev)
    dec = g.FusedDecoder(qm, 6, 16)
    assert not dec.chain
    assert torch.equal(dec.run(idx, 6), g.generate(qm, idx, 6))
