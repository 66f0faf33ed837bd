"""tp_gemm_static_ws with an automatic plan whose splits need more than its 64 MiB: the splits are cut to what fits and the tile
stays, with whole k-tiles and with a k that ends inside one.  The plans are host arithmetic; the products run on the GPU."""
import ctypes

import pytest
import torch

from tests.util import assert_close
from terapipe_amd import _lib as L

CASES = [(L.TP_GEMM_NT, 858, 4368, 40120), (L.TP_GEMM_NT, 534, 10992, 25688), (L.TP_GEMM_NN, 650, 10920, 16896)]


def _desc(op, M, N, K, a=4096, b=4096, c=4096):
    d = L.GemmDesc()
    d.op, d.dtype, d.epilogue, d.M, d.N, d.K = op, L.TP_F16, L.TP_EPI_STORE, M, N, K
    d.A, d.lda, d.B, d.ldb, d.C, d.ldc = a, K, b, (K if op == L.TP_GEMM_NT else N), c, N
    return d


def _tile(d, static_ws):
    v = [ctypes.c_int() for _ in range(3)]
    assert L.load().tp_gemm_tile(ctypes.byref(d), static_ws, *(ctypes.byref(x) for x in v)) == 0
    return tuple(x.value for x in v)


@pytest.mark.parametrize("case", CASES, ids=str)
def test_cut_plans_keep_their_tile(case):
    d = _desc(*case)
    rows, columns, splits = _tile(d, 0)
    assert splits * d.M * d.N * 4 > 64 << 20 and splits == L.load().tp_gemm_splits(ctypes.byref(d))
    r, c, n = _tile(d, 1)
    assert (r, c) == (rows, columns) and 1 <= n < splits and n * d.M * d.N * 4 <= 64 << 20


def test_plans_that_fit_are_those_of_tp_gemm():
    for case in ((L.TP_GEMM_NT, 256, 2048, 8192), (L.TP_GEMM_NN, 2048, 5120, 5120), (L.TP_GEMM_NT, 16, 2048, 2048)):
        assert _tile(_desc(*case), 0) == _tile(_desc(*case), 1)
    forced = _desc(*CASES[0])
    forced.reserved = 7 << 8            # forced splits are not cut (the call is refused)
    assert _tile(forced, 1)[2] == 7


@pytest.mark.gpu
@pytest.mark.parametrize("case", [CASES[0], CASES[2]], ids=str)
def test_cut_products(case):
    op, M, N, K = case
    g = torch.Generator(device="cuda").manual_seed(K)
    a, b = (torch.randn(*s, generator=g, device="cuda").half() for s in ((M, K), (N, K) if op == L.TP_GEMM_NT else (K, N)))
    out = torch.full((M, N), 7.0, dtype=torch.float16, device="cuda")
    d = _desc(op, M, N, K, a.data_ptr(), b.data_ptr(), out.data_ptr())
    L.check(L.load().tp_gemm_static_ws(ctypes.byref(d), torch.cuda.current_stream().cuda_stream), "tp_gemm_static_ws")
    assert_close(out, a.float() @ (b.float().t() if op == L.TP_GEMM_NT else b.float()), torch.float16, "product")
