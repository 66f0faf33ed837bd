"""dQ by workgroups that share their key tiles: what a query's gradient may not depend on."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _dq(q, k, v, o, lse, do, P):
    """dQ alone, forced to the shared form: [BH, T, D]."""
    from terapipe_amd import _lib as L
    from terapipe_amd import ops
    BH, T, D = q.shape
    delta, dqkv = torch.empty(BH, T, device=DEV), torch.full((T, 3 * BH * D), float("nan"), device=DEV, dtype=q.dtype)
    d = ops._attn_desc(q, k, v, o, lse, 1, BH, D, T, P, D ** -0.5)
    d.dq_only, d.reserved2, d.grad_cache_dtype = 1, 32, d.dtype
    d.d_o, d.delta, d.dqkv = do.data_ptr(), delta.data_ptr(), dqkv.data_ptr()
    L.check(L.load().tp_attn_prefix_bwd(ctypes.byref(d), None, 0, ops._stream()), "tp_attn_prefix_bwd")
    return dqkv.view(T, BH, 3, D)[:, :, 0].permute(1, 0, 2)


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("D", [64, 80, 96, 128])
@pytest.mark.parametrize("BH,T,P", [(3, 256, 0), (300, 256, 0), (5, 200, 37), (270, 200, 101), (2, 33, 0)], ids=str)
def test_values_that_a_query_cannot_see(BH, T, P, D, value):
    """An infinite or undefined value in K or V reaches, of the queries before it, at most those of its own block of 32 x 32."""
    from terapipe_amd import ops
    g = torch.Generator(device=DEV).manual_seed(T + P + D)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).half()
    S = P + T
    q, k, v, do = rnd(BH, T, D) * D ** -0.5, rnd(BH, S, D), rnd(BH, S, D), rnd(T, 1, BH * D)
    o, lse = ops.attn_prefix_fwd(q, k, v, 1, BH, D, T, P, D ** -0.5)
    want = _dq(q, k, v, o, lse, do, P)
    assert want.isfinite().all()
    for at in sorted({P + 32, S - 1, P + T // 2, (P + T) // 64 * 64}):
        if not P <= at < S:
            continue
        ends = [P + min(T, t // 32 * 32 + 32) for t in range(T)]
        before = sum(e <= at // 32 * 32 for e in ends)          # queries of blocks that end before the value's block of keys
        for poisoned in (k, v):
            kept = poisoned[:, at].clone()
            poisoned[:, at] = value
            got = _dq(q, k, v, o, lse, do, P)
            poisoned[:, at] = kept
            assert torch.equal(got[:, :before], want[:, :before]), (at, before)
