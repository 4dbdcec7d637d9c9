"""The batched decode head on fp32 operand tiles whose activation planes a
wavefront holds (tiq_decode_linear, TIQ_WF_F32_TILED, up to K = 1280): the same
products in the same order as the row-major weights', so the same bits.
"""
from __future__ import annotations

import pytest
import torch

from gpt2_harness_amd import _lib

pytestmark = pytest.mark.gpu


# units of 32 columns a wavefront: 1..2, 4, 4..5, 5, and 5..6 (the ring)
@pytest.mark.parametrize("M", [5, 33, 64])
@pytest.mark.parametrize("K,N", [(288, 8197), (1024, 16411), (1056, 8225), (1280, 8193), (1312, 8193)])
def test_decode_head_planes_held(dev, M, K, N):
    L = _lib.lib()
    st = torch.cuda.current_stream().cuda_stream
    gen = torch.Generator(device=dev).manual_seed(M + K)
    x, w = torch.randn(M, K, generator=gen, device=dev), torch.randn(N, K, generator=gen, device=dev) * 0.02
    t = torch.empty(int(L.tiq_tile_f32_bytes(N, K)) // 4, device=dev)
    _lib.check(L.tiq_tile_f32(w.data_ptr(), N, K, K, t.data_ptr(), st), "tile f32")

    def head(wt, wf, xr, planes, out, planes_out=None, n=N):
        ws = torch.empty(int(L.tiq_decode_linear_workspace(wf, M, K, n)) + 16, dtype=torch.uint8, device=dev)
        _lib.check(L.tiq_decode_linear(_lib.ptr(xr), K, _lib.ptr(planes), M, K, wt.data_ptr(), wf, None, None, n,
                                       out.data_ptr(), n, None, None, 1e-5, 0, None, 0, None, None, 1e-5,
                                       _lib.ptr(planes_out), ws.data_ptr(), ws.numel() - 16, st), "decode linear")

    planes = torch.zeros(int(L.tiq_decode_planes_bytes(M, K)), dtype=torch.uint8, device=dev)
    eye, xk = torch.eye(K, device=dev), torch.empty(M, K, device=dev)
    head(eye, _lib.WF_F32, x, None, xk, planes, K)  # x times the identity: x and its planes
    assert torch.equal(xk, x)
    y, ref = torch.full((M, N), float("nan"), device=dev), torch.empty(M, N, device=dev)
    head(t, _lib.WF_F32_TILED, None, planes, y)
    head(w, _lib.WF_F32, None, planes, ref)  # N > 8192: one split, the same products in the same order
    assert torch.equal(y, ref)
