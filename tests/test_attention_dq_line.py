"""Which calls take dQ by workgroups that share their key tiles (host code only)."""
import ctypes

import pytest


@pytest.mark.parametrize("pairs,D,T,P", [(24, 64, 1088, 0), (18, 64, 1408, 0), (16, 64, 1536, 0), (13, 64, 1900, 148), (24, 80, 1024, 0), (12, 128, 2048, 0)], ids=str)
def test_calls_with_gradient_caches_too_where_those_for_dq_alone_do(pairs, D, T, P):
    from terapipe_amd import _lib as L
    d = L.AttnDesc()
    d.dtype = d.grad_cache_dtype = L.TP_F16
    d.batch, d.heads, d.head_dim, d.T, d.cache_len, d.cache_rows = 1, pairs, D, T, P, T + P
    for name in ("q", "k_cache", "v_cache", "o", "lse", "d_o", "delta", "dqkv", "dk_cache", "dv_cache"):
        setattr(d, name, 4096)
    for alone in (1, 0):
        d.dq_only, queries = alone, ctypes.c_int(-1)
        assert L.load().tp_attn_bwd_forms(ctypes.byref(d), ctypes.byref(queries), None) == 0
        assert queries.value == 1
