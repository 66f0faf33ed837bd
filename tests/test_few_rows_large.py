"""Which weights above 4096 x 4096 the kernel of a few rows takes where no backward follows (host code only)."""
import ctypes

import pytest


def _rows(M, N, K, reserved):
    """Rows of the launch's tile; 0: the kernel of a few rows, which has none."""
    from terapipe_amd import _lib as L
    d = L.GemmDesc()
    d.op, d.dtype, d.epilogue, d.M, d.N, d.K = L.TP_GEMM_NT, L.TP_F16, L.TP_EPI_STORE, M, N, K
    d.A = d.B = d.C = 4096          # never dereferenced: the plan is host arithmetic on the extents
    d.lda, d.ldb, d.ldc, d.reserved = K, K, N, reserved
    rows, columns, splits = ctypes.c_int(-1), ctypes.c_int(), ctypes.c_int()
    assert L.load().tp_gemm_tile(ctypes.byref(d), 0, ctypes.byref(rows), ctypes.byref(columns), ctypes.byref(splits)) == 0
    return rows.value


@pytest.mark.parametrize("M,N,K,taken", [
    (8, 5120, 5120, True), (8, 20480, 5120, True), (8, 24576, 6144, True), (8, 16384, 16384, True), (8, 15360, 8192, True),
    (8, 12288, 4096, False), (5, 15360, 5120, False), (8, 28672, 4096, False),      # tiles of 64 columns fill their last round
    (4, 12288, 4096, True), (4, 15360, 5120, True), (8, 12288, 2560, True),         # but a LayerNorm's launch is saved
    (4, 4608, 6144, False), (4, 5120, 8192, False), (4, 4096, 16384, True), (4, 5120, 20480, False), (9, 5120, 5120, False)], ids=str)
def test_larger_weights(M, N, K, taken):
    assert (_rows(M, N, K, 1 << 25) == 0) == taken
    assert _rows(M, N, K, 0) > 0            # a backward may follow: tiles, as ever
