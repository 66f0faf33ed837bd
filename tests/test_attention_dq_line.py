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


@pytest.mark.parametrize("D", [64, 80, 96, 128])
def test_rows_beyond_32_bit_offsets_go_elsewhere(D):
    from terapipe_amd import _lib as L
    d = L.AttnDesc()
    d.dtype = d.grad_cache_dtype = L.TP_BF16
    d.batch, d.heads, d.head_dim = 1, 40, D
    for name in ("q", "k_cache", "v_cache", "o", "lse", "d_o", "delta", "dqkv", "dk_cache", "dv_cache"):
        setattr(d, name, 4096)
    queries = ctypes.c_int(-1)
    for rows, want in ((2 ** 30 // D - 512, 1), (2 ** 31 // D, 0), (2 ** 31 // D + 77, 0)):
        for alone, forced in ((1, 0), (0, 0), (1, 32)):
            d.cache_rows, d.T, d.dq_only, d.reserved2 = rows, 2048, alone, forced
            d.cache_len = rows - d.T
            assert L.load().tp_attn_bwd_forms(ctypes.byref(d), ctypes.byref(queries), None) == 0
            assert queries.value == want, (rows, alone, forced)
