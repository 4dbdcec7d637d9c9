"""fp32 activations on the int8 matrix cores (tiq_linear_w8_ws, tiq_linear_w4_ws,
tiq_linear_gelu_in_ws: the rows as four base-256 digit planes, exact int32 sums)
at the sizes where it can go wrong: row counts about its dispatch (65, 127, 128,
129), tile edges in both directions, one k64 step, every pass count of the
digit kernel, the three tiles at their thresholds, the split over K, strided
rows and outputs, and rows of zeros, extremes, infinities and NaN.

Bound against float64, derived: with 2^e <= max|x| the inputs are rounded by at
most 2^(e-30), so sum_k |dx| |w| <= 2^-30 max|x| ||w||_1; the epilogue rounds
three fused steps of sums whose lower digits reach 257 K 2^14, the row factor,
the scale and the bias, each 2^-24 of its value.
"""
from __future__ import annotations

import pytest
import torch

import gpt2_harness_amd as g
from gpt2_harness_amd import _lib

pytestmark = pytest.mark.gpu


def _quantized(K, N, bits, dev, seed):
    gen = torch.Generator(device=dev).manual_seed(seed)
    lin = torch.nn.Linear(K, N, device=dev)
    lin.weight.data = torch.randn(N, K, generator=gen, device=dev) * 0.02
    lin.bias.data = torch.randn(N, generator=gen, device=dev) * 0.1
    return g.quantize_linear(lin, bits)[0], gen


def _call(mod, x, y, K):
    L = _lib.lib()
    M, N = x.shape[0], mod.out_features
    n_ws = int(L.tiq_gemm_w8_workspace(_lib.F32, M, K, N))
    ws = torch.full((max(n_ws, 16),), 0x5A, dtype=torch.uint8, device=x.device)
    fn = L.tiq_linear_w8_ws if mod.fmt == "int8" else L.tiq_linear_w4_ws
    _lib.check(fn(x.data_ptr(), _lib.F32, M, K, x.stride(0), mod.codes.data_ptr(), mod.scale.data_ptr(),
                  _lib.ptr(mod.bias), N, y.data_ptr(), _lib.dtype_code(y.dtype), y.stride(0), ws.data_ptr(), n_ws,
                  torch.cuda.current_stream().cuda_stream), "linear")
    torch.cuda.synchronize()


def _check(mod, x, y, K):
    # codes times scales in 64 bits: the fp32 W_hat carries a rounding of its own
    q = mod.codes if mod.fmt == "int8" else g.unpack_int4(mod.codes, mod.out_features * K).view(-1, K)
    w = q.double() * mod.scale.double().unsqueeze(1)
    ref = x.double() @ w.t() + mod.bias.double()
    top = x.abs().amax(1, keepdim=True).double().clamp(min=2.0**-97)
    u = 2.0**-24
    bound = (top * 2.0**-30 * w.abs().sum(1) * 2
             + 3 * u * top * 2.0**-29 * 257 * K * 2**14 * mod.scale.double()
             + u * (6 * (ref - mod.bias.double()).abs() + 2 * mod.bias.double().abs()))
    err = (y.double() - ref).abs()
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("K,N,M", [
    (64, 128, 65), (768, 3072, 77), (3072, 768, 65), (3072, 768, 127), (1600, 1212, 128), (1024, 37, 129),
    (2048, 132, 160), (4096, 128, 96), (6400, 96, 70), (7232, 128, 130),
    (64, 2048, 2048), (64, 2049, 2047),      # 512 tiles of 64 x 128, and partial ones
    (3200, 1024, 4096), (3200, 1020, 4033),  # 64 x 256 tiles, and partial ones
])
def test_digit_planes(dev, K, N, M, bits):
    mod, gen = _quantized(K, N, bits, dev, K + N + M)
    x = torch.randn(M, K, generator=gen, device=dev)
    x[:, ::97] *= 20.0
    y = torch.full((M, N), float("nan"), device=dev)
    _call(mod, x, y, K)
    _check(mod, x, y, K)
    yb = torch.empty(M, N, device=dev, dtype=torch.bfloat16)
    _call(mod, x, yb, K)
    assert torch.equal(yb, y.bfloat16())


# group-wise int4: groups of one k64 step to the whole row, ragged last groups,
# splits that start inside a group; the bound gains a rounding of the running
# sum a group
@pytest.mark.parametrize("K,N,M,group", [(64, 128, 128, 64), (1600, 1212, 128, 128), (768, 772, 140, 192),
                                         (3072, 768, 65, 128), (3072, 264, 200, 1024), (1600, 2049, 300, 128),
                                         (6400, 96, 70, 320), (2048, 2304, 17, 64), (6400, 1600, 129, 6400)])
def test_digit_planes_groupwise(dev, K, N, M, group):
    gen = torch.Generator(device=dev).manual_seed(K + N + M)
    lin = torch.nn.Linear(K, N, device=dev)
    lin.weight.data = torch.randn(N, K, generator=gen, device=dev) * 0.02
    mod = g.quantize_linear(lin, 4, group_size=group)[0]
    x = torch.randn(M, K, generator=gen, device=dev)
    x[:, ::97] *= 20.0
    y = torch.full((M, N), float("nan"), device=dev)
    L = _lib.lib()
    n_ws = int(L.tiq_gemm_w8_workspace(_lib.F32, M, K, N))
    ws = torch.empty(max(n_ws, 16), dtype=torch.uint8, device=dev)
    for out in (y, yb := torch.empty(M, N, device=dev, dtype=torch.bfloat16)):
        _lib.check(L.tiq_linear_w4g_ws(x.data_ptr(), _lib.F32, M, K, K, mod.codes.data_ptr(), mod.scale.data_ptr(),
                                       group, _lib.ptr(mod.bias), N, out.data_ptr(), _lib.dtype_code(out.dtype), N,
                                       ws.data_ptr(), n_ws, torch.cuda.current_stream().cuda_stream), "linear")
    torch.cuda.synchronize()
    q = g.unpack_int4(mod.codes, N * K).view(N, K)
    s = mod.scale.double().repeat_interleave(group, dim=1)[:, :K]
    w = q.double() * s
    ref = x.double() @ w.t() + mod.bias.double()
    top = x.abs().amax(1, keepdim=True).double()
    u, groups = 2.0**-24, -(-K // group)
    one = w.abs().sum(1)
    bound = (top * 2.0**-30 * one * 2 + 3 * u * top * 2.0**-29 * 257 * K * 2**14 * s.amax(1)
             + (groups + 1) * u * (x.double().abs() @ w.abs().t()) + 8 * u * (ref.abs() + mod.bias.double().abs()))
    err = (y.double() - ref).abs()
    assert bool((err <= bound).all()), float((err / bound).max())
    assert torch.equal(yb, y.bfloat16())


# Groups to either side of the 256 columns whose digit sums join in int32, with
# nothing that cancels: constant rows whose digits are (lowest first) (-128, 103,
# 102, 38), (0, 0, 0, 32) and (-128, 21, -82, 64), weights of one sign, so every
# digit sum is as large as its group makes it. Bound: the inputs' 2^-30, a rounding
# of the running sum a group and a split (at least six k64 steps each) and six more.
@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("K,N,M,group", [(1024, 128, 128, 256), (960, 128, 129, 320), (1024, 1056, 130, 512),
                                         (1024, 128, 128, 1024), (3072, 4096, 256, 3072), (3072, 136, 66, 1536),
                                         (6400, 96, 70, 6400)])
def test_digit_planes_wide_groups_of_one_sign(dev, K, N, M, group, sign):
    lin = torch.nn.Linear(K, N, device=dev)
    lin.weight.data = (torch.rand(N, K, device=dev) * 0.01 + 0.99) * sign
    lin.weight.data[: N // 2] = sign  # every code at its extreme
    lin.bias.data.zero_()
    mod = g.quantize_linear(lin, 4, group_size=group)[0]
    x = torch.tensor([1.2, 1.0, 1.99], device=dev)[torch.arange(M, device=dev) % 3].unsqueeze(1).repeat(1, K)
    with torch.no_grad():
        y = mod(x)
    q = g.unpack_int4(mod.codes, N * K).view(N, K)
    w = q.double() * mod.scale.double().repeat_interleave(group, dim=1)[:, :K]
    ref = x.double() @ w.t()
    bound = ref.abs() * (2.0**-29 + (-(-K // group) + K // 384 + 6) * 2.0**-24)
    err = (y.double() - ref).abs()
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("bits", [8, 4])
def test_digit_planes_strided(dev, bits):
    K, N, M = 768, 772, 140
    mod, gen = _quantized(K, N, bits, dev, 5)
    x = torch.randn(M, K + 12, generator=gen, device=dev)[:, :K]
    full = torch.full((M, N + 3), 7.0, device=dev)
    _call(mod, x, full[:, :N], K)
    _check(mod, x, full[:, :N], K)
    assert bool((full[:, N:] == 7.0).all())


def test_digit_planes_extreme_rows(dev):
    K, N, M = 768, 256, 128
    mod, gen = _quantized(K, N, 8, dev, 6)
    x = torch.randn(M, K, generator=gen, device=dev)
    x[0] = 0.0
    x[1] *= 1e30
    x[2] *= 1e-36
    x[3] *= 1e-44  # subnormal inputs
    x[4, 5] = 3e4  # one element far above the rest
    y = torch.empty(M, N, device=dev)
    _call(mod, x, y, K)
    _check(mod, x, y, K)
    assert torch.equal(y[0], mod.bias.data)
    bad = x.clone()
    bad[7, 3], bad[9, 700], bad[11, 0] = float("inf"), float("nan"), float("-inf")
    yb = torch.empty(M, N, device=dev)
    _call(mod, bad, yb, K)
    for m in (7, 9, 11):
        assert bool(yb[m].isnan().all())
    keep = [m for m in range(M) if m not in (7, 9, 11)]
    assert torch.equal(yb[keep], y[keep])


# Past the 65536 columns whose digit sums fit int32: three bf16 planes and the bf16
# GEMMs (the staged one; the LDS one for groups). Bound: one rounding a product of
# the three planes' sums in the worst order, two more an output.
@pytest.mark.parametrize("fmt", ["int8", "int4", "g128"])
@torch.no_grad()
def test_columns_past_the_digit_sums(dev, fmt):
    K, N, M = 65664, 96, 130
    gen = torch.Generator(device=dev).manual_seed(3)
    lin = torch.nn.Linear(K, N, device=dev)
    lin.weight.data = torch.randn(N, K, generator=gen, device=dev) * 0.02
    mod = g.quantize_linear(lin, 8 if fmt == "int8" else 4, group_size=128 if fmt == "g128" else None)[0]
    if fmt == "int8":
        w = mod.codes.double() * mod.scale.double().unsqueeze(1)
    else:
        w = g.unpack_int4(mod.codes, N * K).view(N, K).double()
        w *= mod.scale.double().repeat_interleave(128, dim=1) if fmt == "g128" else mod.scale.double().unsqueeze(1)
    x = torch.randn(M, K, generator=gen, device=dev)
    x[:, ::97] *= 1e4  # nothing is held relative to the row's largest
    for y, v in ((mod(x), x), (mod.forward_gelu_in(x), g.model.gelu_tanh(x))):
        ref = v.double() @ w.t() + mod.bias.double()
        err = (y.double() - ref).abs()
        work = v.double().abs() @ w.abs().t() + mod.bias.double().abs()
        assert bool((err <= (K + 2) * 2.0**-24 * work).all())
        assert err.norm() <= 3.0 * K**0.5 * 2.0**-24 * ref.norm()
