"""The deep rings of 64 x 32, 64 x 64 and 64 x 128 tiles (tile configuration 12 on weights of up to 4096 x 4096) against the fp64 product:
the tiles the estimate picks (tails of k, rows and columns that end inside a tile, k splits), and each width forced: k-tiles of 128
below, at and above its stage count (6, 5 and 3), rings that wrap several times, k that ends inside a k-tile, splits of unequal
length."""
import ctypes

import pytest
import torch

from tests.util import assert_close

DEV = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("op", ["NT", "NN"])
@pytest.mark.parametrize("M,N,K,ksplit", [
    (33, 8, 8, 1), (64, 32, 128, 1), (65, 40, 136, 1), (100, 264, 640, 1), (200, 1000, 776, 1),
    (64, 1024, 2056, 3),
    (256, 4800, 1600, 1), (200, 4000, 392, 1),
    (512, 4096, 264, 1), (500, 3000, 1000, 1), (256, 4000, 1160, 3), (130, 2048, 2048, 5),
], ids=str)
def test_deep_rings(op, M, N, K, ksplit, dtype):
    from terapipe_amd import _lib as L
    from terapipe_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M + 3 * N + 7 * K)
    A = torch.randn(M, K, generator=g, device=DEV).to(dtype)
    B = (torch.randn((N, K) if op == "NT" else (K, N), generator=g, device=DEV) * 0.1).to(dtype)
    bias = torch.randn(N, generator=g, device=DEV).to(dtype)
    res = torch.randn(M, N, generator=g, device=DEV).to(dtype)
    out = torch.full((M + 2, N), 77.0, dtype=dtype, device=DEV)
    ops.gemm(L.TP_GEMM_NT if op == "NT" else L.TP_GEMM_NN, A, B, M, N, K, C=out[1:M + 1], epilogue=L.TP_EPI_BIAS_RESIDUAL,
             bias=bias, residual=res, tile_cfg=12, ksplit=ksplit)
    ref = A.double() @ (B.double().t() if op == "NT" else B.double()) + bias.double() + res.double()
    assert_close(out[1:M + 1], ref, dtype, "%s %dx%dx%d" % (op, M, N, K))
    assert bool((out[0] == 77.0).all()) and bool((out[M + 1] == 77.0).all())


# nk k-tiles: 1, 2, 3, 5, 6, 7 and 16; splits of 6 + 6 + 5, 13 + 12 and 3 + 3 + 3 + 1 k-tiles
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("op", ["NT", "NN"])
@pytest.mark.parametrize("columns", [32, 64, 128])
@pytest.mark.parametrize("M,N,K,ksplit", [
    (33, 8, 104, 1), (65, 40, 136, 1), (100, 264, 384, 1), (64, 128, 640, 1), (33, 72, 768, 1), (130, 200, 776, 1), (70, 136, 1992, 1),
    (130, 264, 2056, 3), (200, 1000, 3080, 2), (65, 136, 1160, 4)], ids=str)
def test_every_width(columns, M, N, K, ksplit, op, dtype):
    from terapipe_amd import _lib as L
    from terapipe_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M + 3 * N + 7 * K)
    A = torch.randn(M, K, generator=g, device=DEV).to(dtype)
    B = (torch.randn((N, K) if op == "NT" else (K, N), generator=g, device=DEV) * 0.1).to(dtype)
    out = torch.full((M + 2, N), 77.0, dtype=dtype, device=DEV)
    sink = []
    ops.gemm(L.TP_GEMM_NT if op == "NT" else L.TP_GEMM_NN, A, B, M, N, K, C=out[1:M + 1], tile_cfg=12, ksplit=ksplit | columns << 8,
             desc_sink=sink)
    rows, cols, splits = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    assert L.load().tp_gemm_tile(ctypes.byref(sink[0]), 0, ctypes.byref(rows), ctypes.byref(cols), ctypes.byref(splits)) == 0
    assert (rows.value, cols.value, splits.value) == (64, columns, ksplit)
    ref = A.double() @ (B.double().t() if op == "NT" else B.double())
    assert_close(out[1:M + 1], ref, dtype, "%s %dx%dx%d, %d columns" % (op, M, N, K, columns))
    assert bool((out[0] == 77.0).all()) and bool((out[M + 1] == 77.0).all())
