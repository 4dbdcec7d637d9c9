"""The fp32 head over every position of a batch (tiq_linear_f32_ws, GPT.forward).

Error bound against float64, derived: six fp32 roundings per 16 columns plus the
dropped plane products (three of at most 2^-24 of their product), (K + 8) 2^-24
sum |x| |w| in the worst order; in the 2-norm it may not exceed a plain fp32
GEMM's by more than an eighth.
"""
from __future__ import annotations

import pytest
import torch

import gpt2_harness_amd as g
from gpt2_harness_amd import _lib

pytestmark = pytest.mark.gpu


def _call(x, w, y, ws=None):
    L = _lib.lib()
    M, K = x.shape
    N = w.shape[0]
    need = int(L.tiq_linear_f32_workspace(M, K, N))
    if ws is None:
        ws = torch.empty(max(need, 16), dtype=torch.uint8, device=x.device)
    return L.tiq_linear_f32_ws(x.data_ptr(), M, K, x.stride(0), w.data_ptr(), w.stride(0), N, y.data_ptr(),
                               y.stride(0), ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)


# Rows and columns at and beside whole 128-wide tiles and 32-row blocks, odd
# output strides, one unit of 32 columns and odd counts of units.
@pytest.mark.parametrize("M,K,N", [(65, 768, 50257), (66, 32, 4096), (127, 96, 4097), (128, 1024, 4224),
                                   (129, 1280, 4225), (300, 1600, 5003), (512, 768, 8191), (1024, 64, 4100)])
def test_head_over_a_batch(dev, M, K, N):
    gen = torch.Generator(device=dev).manual_seed(M + K + N)
    x = torch.randn(M, K + 4, generator=gen, device=dev)[:, :K]
    x[:, :: max(1, K // 3)] *= 8.0
    w = torch.randn(N, K, generator=gen, device=dev) * 0.02
    y = torch.full((M + 1, N), float("nan"), device=dev)
    assert _call(x, w, y[:M]) == _lib.OK
    assert torch.isnan(y[M]).all()
    ref = x.double() @ w.double().t()
    err = (y[:M].double() - ref).abs()
    assert bool((err <= (K + 8) * 2.0**-24 * (x.double().abs() @ w.double().abs().t())).all())
    assert err.norm() <= 1.125 * ((x @ w.t()).double() - ref).norm() + 1e-30


@pytest.mark.parametrize("M,K,N", [(65, 96, 4097), (130, 768, 4224)])
def test_head_of_infinities(dev, M, K, N):
    """Infinities, NaN and values that round to infinity in bf16 mean in x and w what
    they mean in an fp32 sum; other outputs do not notice."""
    gen = torch.Generator(device=dev).manual_seed(M)
    x = torch.randn(M, K, generator=gen, device=dev)
    w = torch.randn(N, K, generator=gen, device=dev) * 0.02
    w[5::7, 3] = 0.0  # inf times zero
    plain, y = torch.empty(M, N, device=dev), torch.empty(M, N, device=dev)
    assert _call(x, w, plain) == _lib.OK
    inf, top = float("inf"), torch.finfo(torch.float32).max
    for m, v in ((0, inf), (7, -inf), (33, float("nan")), (40, top), (41, 3.393e38), (M - 1, -3.4e38)):
        x[m, 3] = v
    for n, v in ((2, -inf), (100, 1e30), (4096, top)):
        w[n, K - 1] = v
    assert _call(x, w, y) == _lib.OK
    ref = (x.double() @ w.double().t()).float()  # past fp32's range: infinite
    finite = x.isfinite().all(1, keepdim=True) & w.isfinite().all(1)
    assert torch.equal(y.isnan(), ref.isnan())
    assert torch.equal(y[~finite & ~ref.isnan()], ref[~finite & ~ref.isnan()])
    work = x.double().abs() @ w.double().abs().t()
    ok = finite & (work < top)
    assert bool(((y.double() - ref.double()).abs() <= (K + 8) * 2.0**-24 * work)[ok].all())
    rows = [m for m in range(M) if m not in (0, 7, 33, 40, 41, M - 1)]
    cols = [n for n in range(N) if n not in (2, 100, 4096)]
    assert torch.equal(y[rows][:, cols], plain[rows][:, cols])


def test_head_refusals(dev):
    x, w, y = (torch.zeros(s, device=dev) for s in ((65, 64), (4096, 64), (65, 4096)))
    L = _lib.lib()
    assert L.tiq_linear_f32_workspace(64, 64, 4096) == 0 and L.tiq_linear_f32_workspace(65, 48, 4096) == 0
    assert _call(x[:64], w, y[:64]) == _lib.EUNSUPPORTED
    assert _call(x, w[:4095], y[:, :4095]) == _lib.EUNSUPPORTED
    assert _call(x, w, y, torch.empty(1024, dtype=torch.uint8, device=dev)) == _lib.EWORKSPACE
    assert _call(torch.zeros(65 * 64 + 1, device=dev)[1:].view(65, 64), w, y) == _lib.EALIGN
    assert _call(x[:0], w, y[:0]) == _lib.OK


def test_model_logits_and_where_the_module_runs(dev):
    cfg = g.GPTConfig(vocab_size=5003, n_layer=1, n_head=4, n_embd=256)
    torch.manual_seed(0)
    model = g.GPT(cfg).to(dev).eval()
    idx = torch.randint(0, 5003, (2, 50), device=dev)
    seen = []
    with torch.no_grad():
        y = model(idx)["logits"]
        handle = model.lm_head.register_forward_hook(lambda *a: seen.append(1))
        ref = model(idx)["logits"]
        handle.remove()
        assert seen and y.shape == ref.shape
        assert ((y - ref).double().norm() / ref.double().norm()).item() <= 2.0**-20
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert model(idx)["logits"].dtype == torch.bfloat16
    assert model(idx)["logits"].requires_grad
