"""Products of a few rows that sum in another order are for calls that no backward follows: half a rounding more or less in a forward
that one does follow turns ReLU units near zero on or off, and the gradients behind them move."""
import ctypes

import pytest
import torch

from terapipe_amd import _lib, ops
from terapipe_amd import _layer_core as core


def _splits(M, N, K, reserved):
    d = _lib.GemmDesc()
    d.op, d.dtype, d.epilogue, d.M, d.N, d.K = _lib.TP_GEMM_NT, _lib.TP_F16, _lib.TP_EPI_STORE, M, N, K
    d.A = d.B = d.C = 4096          # never dereferenced: the plan is host arithmetic on the extents
    d.lda, d.ldb, d.ldc, d.reserved = K, K, N, reserved
    return _lib.load().tp_gemm_splits(ctypes.byref(d))


@pytest.mark.parametrize("M,N,K", [(4, 2048, 8192), (8, 1024, 8192), (1, 2048, 8192)], ids=str)
def test_k_splits(M, N, K):
    assert _splits(M, N, K, 0) > 1 and _splits(M, N, K, 1 << 25) == 1
    assert _splits(9, N, K, 1 << 25) == _splits(9, N, K, 0)


def test_who_says_that_no_backward_follows(monkeypatch):
    """The forward-only stack, by one buffer for both LayerNorms' rows; a layer on its own gives the same bits with and without autograd."""
    made = []
    monkeypatch.setattr(core, "layers_fwd", lambda images, n, device: made.append(_lib.LayerDesc.from_buffer_copy(images[-len(images) // n:])))
    monkeypatch.setattr(ops, "_require_cuda", lambda *tensors: None)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    import terapipe_amd as ta
    layer = ta.ModelParallelTransformerLayer(64, 128, 1, device="cpu")
    x = torch.zeros(4, 1, 64)
    stack = ta.TransformerLayers(2, 64, 128, 1, dtype=torch.float32, device="cpu")
    with torch.no_grad():
        stack(x, stack.create_cache(1, 4), 0)
        layer(x)
    layer(x.requires_grad_())
    assert [d.xn == d.hn for d in made] == [True, False, False]
