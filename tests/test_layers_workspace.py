"""The workspace that a chain of layers asks for holds the largest of its layers' (host code only)."""
import ctypes

import pytest


def _layer(no_backward, hidden=2048, cache_len=0):
    from terapipe_amd import _lib as L
    d = L.LayerDesc()
    d.dtype, d.T, d.batch, d.heads, d.hidden, d.ffn, d.cache_len, d.cache_rows = L.TP_F16, 1, 4, 16, hidden, 4 * hidden, cache_len, cache_len + 1
    for i in range(12):
        d.w[i] = 4096               # never dereferenced: the plan is host arithmetic
    for name, kind in d._fields_:
        if kind is ctypes.c_void_p:
            setattr(d, name, 4096)
    d.no_backward = no_backward
    return d


def _need(*layers):
    from terapipe_amd import _lib as L
    a = (L.LayerDesc * len(layers))(*layers)
    return L.load().tp_layers_fwd_workspace_bytes(ctypes.addressof(a), len(layers))


@pytest.mark.parametrize("order", [(0, 1), (1, 0), (1, 1, 0), (0, 0, 1)])
def test_layers_with_and_without_a_backward(order):
    alone = {n: _need(_layer(n)) for n in (0, 1)}
    assert alone[0] > alone[1]      # k splits, which the forms of a few rows without a backward do not need
    assert _need(*(_layer(n) for n in order)) == alone[0]
