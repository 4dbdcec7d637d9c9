"""Row counts between the decode kernels and the prefill GEMM (5 .. 127) through
QuantLinear: bf16 rows that the MFMA GEMM takes below 128 (about its thresholds
in rows and in product size, split over K for a long K) and fp32 rows that the
digit planes take, for every weight format.

Bound against float64, derived: the result's own rounding (bf16: 2^-9 of it) and
one fp32 rounding a product of the sum (K + 2 of them, group-wise one more a
group), 2^-24 sum |x| |w| each in the worst order.
"""
from __future__ import annotations

import pytest
import torch

import gpt2_harness_amd as g

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ["int8", "int4", "int4_groupwise"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("K,N,M", [
    (768, 768, 16), (768, 768, 23), (768, 768, 24), (768, 2304, 7), (768, 2304, 8), (768, 2304, 65), (1600, 4800, 9),
    (6400, 1600, 9), (6400, 1600, 10), (6400, 1600, 17), (6400, 1600, 32), (3072, 768, 64), (3136, 768, 17),
    (1600, 1600, 33), (1536, 776, 127), (768, 770, 66), (800, 768, 70),  # N and K the GEMMs do not take
])
def test_rows_below_the_prefill(dev, K, N, M, dtype, fmt):
    gen = torch.Generator(device=dev).manual_seed(K + N + M)
    lin = torch.nn.Linear(K, N, device=dev)
    lin.weight.data = torch.randn(N, K, generator=gen, device=dev) * 0.02
    mod = g.quantize_linear(lin, 8 if fmt == "int8" else 4, group_size=128 if fmt == "int4_groupwise" else None)[0]
    assert mod.fmt == fmt
    x = torch.randn(M, K, generator=gen, device=dev).to(dtype)
    with torch.no_grad():
        y = mod(x)
        assert torch.equal(mod(x), y)
    w = mod.weight.double()
    ref = x.double() @ w.t() + mod.bias.double()
    work = x.double().abs() @ w.abs().t() + mod.bias.double().abs()
    bound = work * (K + 54) * 2.0**-24 + (ref.abs() * 2.0**-8 if dtype == torch.bfloat16 else 0.0)
    assert bool(((y.double() - ref).abs() <= bound).all())
