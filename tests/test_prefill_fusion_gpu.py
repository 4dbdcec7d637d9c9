"""The Linears of a prompt's block with their LayerNorm, residual and cache
writes (tiq_linear_prefill_ws, QuantLinear.forward_prefill, Block.forward).

Residual and cache writes must equal, bit for bit, the plain product followed by
the add or the copies; the LayerNorm, whose statistics are summed in another
order than torch's, is held to a float64 restatement. A block that runs fused
must agree with the same block run module by module (a hook forces that).
"""
from __future__ import annotations

import pytest
import torch

import gpt2_harness_amd as g
from gpt2_harness_amd import _lib
from gpt2_harness_amd.model import Block, CausalSelfAttention, KVCache

pytestmark = pytest.mark.gpu

FORMATS = {"int8": {"bits": 8}, "int4": {"bits": 4}, "g128": {"bits": 4, "group_size": 128}}


def _linear(K, N, fmt, dev, seed=0):
    gen = torch.Generator().manual_seed(seed + K + N)
    lin = torch.nn.Linear(K, N)
    lin.weight.data = torch.randn(N, K, generator=gen) * 0.02
    lin.bias.data = torch.randn(N, generator=gen) * 0.1
    o = FORMATS[fmt]
    return g.quantize_linear(lin.to(dev), o["bits"], group_size=o.get("group_size"))[0].to(dev)


def _ln(C, dev):
    gen = torch.Generator().manual_seed(C)
    ln = torch.nn.LayerNorm(C)
    ln.weight.data = 1.0 + 0.1 * torch.randn(C, generator=gen)
    ln.bias.data = 0.1 * torch.randn(C, generator=gen)
    return ln.to(dev)


def _rows(M, K, dev, seed=1):
    gen = torch.Generator().manual_seed(seed + M)
    x = torch.randn(M, K, generator=gen)
    x[:, :: K // 3] *= 8.0
    return x.to(dev)


def _rel(a, b):
    return ((a.double() - b).norm() / b.norm()).item()


# Rows at the edges of 8-row LayerNorm groups and 32- and 64-row tiles; widths
# of one and two register passes with a ragged last one (1600 = 1024 + 576); the
# small, the persistent and (K = 6400, M = 4100) the wide product tile; K splits.
SHAPES = [(65, 768, 2304), (96, 1600, 1600), (129, 1024, 3072), (600, 2048, 256), (1001, 1600, 4800)]


@pytest.mark.parametrize("fmt", sorted(FORMATS))
@pytest.mark.parametrize("M,K,N", SHAPES)
@torch.no_grad()
def test_layer_norm_in(dev, fmt, M, K, N):
    lin, ln, x = _linear(K, N, fmt, dev), _ln(K, dev), _rows(M, K, dev) + 3.0
    y = lin.forward_prefill(x, ln=ln)
    assert y is not None
    x64 = torch.nn.functional.layer_norm(x.double(), (K,), ln.weight.double(), ln.bias.double(), ln.eps)
    ref = x64 @ lin.weight.double().t() + lin.bias.double()
    # a LayerNorm's handful of fp32 roundings (2^-24 each, at a mean of three
    # deviations), against torch's own through the plain product
    assert _rel(y, ref) <= max(1.25 * _rel(lin(ln(x)), ref), 2.0**-21)


@pytest.mark.parametrize("fmt", sorted(FORMATS))
@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("M,K,N", [*SHAPES, (77, 3072, 768), (4100, 6400, 1600)])
@torch.no_grad()
def test_residual_out(dev, fmt, gelu, M, K, N):
    lin, x, res = _linear(K, N, fmt, dev), _rows(M, K, dev), _rows(M, N, dev, 2)
    y = lin.forward_prefill(x, gelu=gelu, residual=res)
    assert y is not None
    plain = lin(g.model.gelu_tanh(x) if gelu else x)
    assert torch.equal(y, res + plain)
    assert torch.equal(lin.forward_prefill(x, gelu=gelu), plain)


@pytest.mark.parametrize("fmt", sorted(FORMATS))
@pytest.mark.parametrize("B,T,first,C", [(65, 1, 3, 768), (3, 43, 0, 768), (1, 1001, 0, 1024), (9, 128, 5, 1600),
                                         (33, 31, 0, 1280)])
@torch.no_grad()
def test_keys_and_values_into_the_cache(dev, fmt, B, T, first, C):
    H = C // 64
    lin, x = _linear(C, 3 * C, fmt, dev), _rows(B * T, C, dev)
    # slots inside a larger buffer: what lies around them stays
    big = torch.full((2, B, H, first + T + 2, 64), -7.0, device=dev)
    k, v = (big[i, :, :, first : first + T] for i in (0, 1))
    q = lin.forward_prefill(x, kv=(k, v, T))
    assert q is not None
    ref = lin(x).view(B, T, 3, H, 64).permute(2, 0, 3, 1, 4)
    assert torch.equal(q.view(B, T, H, 64).transpose(1, 2), ref[0])
    assert torch.equal(k, ref[1]) and torch.equal(v, ref[2])
    assert (big[:, :, :, :first] == -7.0).all() and (big[:, :, :, first + T :] == -7.0).all()


def _block(fmt, dev, C=768, dropout=0.0):
    cfg = g.GPTConfig(vocab_size=64, n_layer=1, n_head=C // 64, n_embd=C, dropout=dropout)
    torch.manual_seed(0)
    blk = Block(cfg).to(dev)
    for owner, name, (k, n) in ((blk.attn, "c_attn", (C, 3 * C)), (blk.attn, "c_proj", (C, C)),
                                (blk.mlp, "c_fc", (C, 4 * C)), (blk.mlp, "c_proj", (4 * C, C))):
        setattr(owner, name, _linear(k, n, fmt, dev))
    blk.ln_1, blk.ln_2 = _ln(C, dev), _ln(C, dev)
    return blk.eval()


@pytest.mark.parametrize("fmt", sorted(FORMATS))
@pytest.mark.parametrize("B,T,cut,C", [(1, 8, 8, 768), (2, 37, 20, 768), (4, 128, 128, 768), (1, 301, 150, 1600)])
@torch.no_grad()
def test_block_fused_and_by_modules(dev, fmt, B, T, cut, C):
    blk, x = _block(fmt, dev, C), _rows(B * T, C, dev).view(B, T, C)
    seen = []

    def run():
        cache = KVCache(1)  # grows by itself
        y = [blk(x[:, :cut].contiguous(), cache)] + ([blk(x[:, cut:].contiguous(), cache)] if cut < T else [])
        return torch.cat(y, 1), cache.keys[0], cache.values[0]

    fused = run()
    handle = blk.ln_1.register_forward_hook(lambda *a: seen.append(1))
    plain = run()
    handle.remove()
    assert seen and torch.equal(x, _rows(B * T, C, dev).view(B, T, C))
    for a, b in zip(fused, plain):
        assert a.shape == b.shape
        # both are a few fp32 roundings from the exact block: 2^-20 covers the sum
        assert _rel(a, b.double()) <= 2.0**-20


def test_block_keeps_modules_where_it_must(dev):
    blk, x = _block("int8", dev), _rows(256, 768, dev).view(2, 128, 768)
    with torch.no_grad():
        assert blk._prefill(x, None) is not None
        assert blk._prefill(x[:, ::2], None) is None          # rows with gaps
        assert blk._prefill(x.bfloat16(), None) is None
        assert blk._prefill(x[:1, :4].contiguous(), None) is None  # decode-sized
        blk.mlp.c_fc.forward = lambda t: t                     # replaced by a caller
        assert blk._prefill(x, None) is None
        del blk.mlp.c_fc.forward
    assert blk._prefill(x, None) is None                       # the LayerNorms want gradients
    y = blk(x.clone().requires_grad_())
    assert y.requires_grad


@torch.no_grad()
def test_attention_falls_back_to_copies(dev):
    """A cache that the kernel may not write (16-bit buffers) is filled by copies."""
    blk = _block("int8", dev)
    x = _rows(128, 768, dev).view(1, 128, 768)
    half = KVCache.over([torch.zeros(1, 12, 130, 64, device=dev, dtype=torch.bfloat16)],
                        [torch.zeros(1, 12, 130, 64, device=dev, dtype=torch.bfloat16)])
    assert half._append_slots(0, 1, 12, 128, x) is None
    full = KVCache.over([torch.zeros(1, 12, 130, 64, device=dev)], [torch.zeros(1, 12, 130, 64, device=dev)])
    y = CausalSelfAttention.forward(blk.attn, x, full)
    ref = blk.attn(x)  # no cache: the product's own rows
    assert torch.equal(y, ref) and full.length(0) == 128


class _Recording(KVCache):
    def update(self, layer, k, v):
        self.seen = getattr(self, "seen", 0) + k.shape[-2]
        return super().update(layer, k, v)


class _Duck:
    """The members a forward pass uses, and no others."""

    def __init__(self):
        self.inner, self.seen = KVCache(1), 0

    @property
    def seq_len(self):
        return self.inner.seq_len

    def length(self, layer):
        return self.inner.length(layer)

    def update(self, layer, k, v):
        self.seen += k.shape[-2]
        return self.inner.update(layer, k, v)


@torch.no_grad()
def test_caches_with_an_update_of_their_own(dev):
    blk = _block("int8", dev)
    x = _rows(128, 768, dev).view(1, 128, 768)
    plain = KVCache(1)
    want = blk(x, plain)
    patched, seen = KVCache(1), []
    update = patched.update
    patched.update = lambda layer, k, v: (seen.append(k.shape[-2]), update(layer, k, v))[1]
    for cache in (_Recording(1), _Duck(), patched):
        y = blk(x, cache)
        inner = getattr(cache, "inner", cache)
        assert (sum(seen) if cache is patched else cache.seen) == 128 and cache.length(0) == 128
        assert torch.equal(inner.keys[0], plain.keys[0]) and torch.equal(inner.values[0], plain.values[0])
        assert torch.equal(y, want)
        assert torch.equal(CausalSelfAttention.forward(blk.attn, x, type(cache)() if cache.__class__ is _Duck
                                                       else type(cache)(1)), blk.attn(x))


@torch.no_grad()
def test_no_attempt_where_the_product_is_split(dev, monkeypatch):
    """The attention asks before it makes room and calls: a product split over K, or
    rows that are not its, would refuse the cache writes."""
    calls = []
    real = g.QuantLinear.forward_prefill
    monkeypatch.setattr(g.QuantLinear, "forward_prefill", lambda self, *a, **k: (calls.append(1), real(self, *a, **k))[1])
    for fmt, C, M, takes in (("g128", 1600, 24, False), ("g128", 1600, 300, True), ("int8", 768, 24, False),
                             ("int8", 768, 65, True), ("int4", 1600, 129, True)):
        blk, x = _block(fmt, dev, C), _rows(M, C, dev).view(1, M, C)
        cache = KVCache(1)
        assert blk.attn.c_attn.writes_kv(M) == takes
        calls.clear()
        y = blk.attn(x, cache)
        assert len(calls) == takes and cache.length(0) == M
        k, v = (torch.zeros(1, C // 64, M, 64, device=dev) for _ in range(2))
        assert (real(blk.attn.c_attn, x.view(M, C), kv=(k, v, M)) is not None) == takes
        assert _rel(y, blk.attn(x).double()) <= 2.0**-20


def test_arguments(dev):
    lin = _linear(768, 2304, "int8", dev)
    L, M, K, N = _lib.lib(), 128, 768, 2304
    st = torch.cuda.current_stream().cuda_stream
    x, y, ln = _rows(M, K, dev), torch.empty(M, N, device=dev), _ln(K, dev)
    res, kv = torch.zeros(M, N, device=dev), torch.zeros(2, 1, 12, M, 64, device=dev)
    need = int(L.tiq_linear_workspace(_lib.WF_INT8, _lib.F32, M, K, N))
    ws = torch.empty(need, dtype=torch.uint8, device=dev)

    def call(m=M, wf=_lib.WF_INT8, lw=None, lb=None, gelu=0, r=None, ldr=0, k=None, v=None, T=0, ws_bytes=need, ldy=N):
        return L.tiq_linear_prefill_ws(x.data_ptr(), m, K, K, lin.codes.data_ptr(), wf, lin.scale.data_ptr(), None, 0,
                                       _lib.ptr(lin.bias), N, y.data_ptr(), ldy, lw, lb, 1e-5, gelu, r, ldr, k, v,
                                       12 * M * 64, M * 64, 64, T, ws.data_ptr(), ws_bytes, st)

    w, b, k, v = ln.weight.data_ptr(), ln.bias.data_ptr(), kv[0].data_ptr(), kv[1].data_ptr()
    assert call() == _lib.OK
    assert call(m=0) == _lib.OK
    assert call(m=8) == _lib.EUNSUPPORTED
    assert call(wf=_lib.WF_F32) == _lib.EINVAL
    assert call(lw=w) == _lib.EINVAL
    assert call(lw=w, lb=b, gelu=1) == _lib.EINVAL
    assert call(r=res.data_ptr(), ldr=N - 1) == _lib.EINVAL
    assert call(r=res.data_ptr(), ldr=N, k=k, v=v, T=M) == _lib.EINVAL
    assert call(k=k, T=M) == _lib.EINVAL
    assert call(k=k, v=v, T=0) == _lib.EINVAL
    assert call(k=k, v=v, T=100) == _lib.EINVAL  # not whole sequences
    assert call(ldy=K - 1) == _lib.EINVAL
    assert call(ws_bytes=4096) == _lib.EWORKSPACE
    assert call(k=k, v=v, T=M, ldy=K) == _lib.OK
    torch.cuda.synchronize()
