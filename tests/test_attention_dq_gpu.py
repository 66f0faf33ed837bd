"""dQ by workgroups that share their key tiles: what a query's gradient may not depend on."""
import ctypes

import pytest
import torch

from tests.util import assert_close

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
@pytest.mark.parametrize("BH,T,P", [(3, 256, 0), (300, 256, 0), (5, 200, 37), (270, 200, 101), (2, 33, 0), (27, 1411, 0)], ids=str)
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


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("D", [64, 80, 96, 128])
@pytest.mark.parametrize("BH,T,P", [(25, 1400, 0), (27, 1411, 705), (32, 1473, 100), (24, 1536, 0), (33, 1399, 0), (43, 1500, 13)], ids=str)
def test_long_sequences_of_few_heads(BH, T, P, D, dtype):
    """Both sides of the lines between the eight-wave form and the two others, with key tiles and query blocks that end inside."""
    from terapipe_amd import ops
    g = torch.Generator(device=DEV).manual_seed(T + P + D)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    S, sc = P + T, D ** -0.5
    q, k, v, do = rnd(BH, T, D) * sc, rnd(BH, S + 3, D), rnd(BH, S + 3, D), rnd(T, 1, BH * D)
    k[:, S:], v[:, S:] = float("nan"), float("nan")         # rows past the slice are never used
    o, lse = ops.attn_prefix_fwd(q, k, v, 1, BH, D, T, P, sc)
    got = _dq(q, k, v, o, lse, do, P).double()
    unseen = torch.arange(S, device=DEV)[None] > P + torch.arange(T, device=DEV)[:, None]
    for h in range(BH):
        kd, vd, dod, od = k[h, :S].double(), v[h, :S].double(), do[:, 0, h * D:(h + 1) * D].double(), o[:, 0, h * D:(h + 1) * D].double()
        p = torch.softmax((q[h].double() @ kd.t()).masked_fill(unseen, float("-inf")), -1)
        want = (p * (dod @ vd.t() - (od * dod).sum(-1, keepdim=True))) @ kd * sc
        assert_close(got[h], want, dtype, "dq of head %d" % h)


@pytest.mark.parametrize("D", [80, 128])
def test_keys_beyond_4_gib(D):
    """A head whose K and V rows are more than 4 GiB each: two rows near the end take all of a query's weight but what 16 million
    zeros share."""
    S = ((1 << 32) // (2 * D) // 32 + 4) * 32
    k, v = (torch.zeros(1, S, D, device=DEV, dtype=torch.float16) for _ in range(2))
    g = torch.Generator(device=DEV).manual_seed(D)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    T, P, sc, far = 1, S - 1, D ** -0.5, [S - 70, S - 1]
    q = (rnd(1, T, D) * 0.5).half()
    for at, score in zip(far, (20.0, 21.0)):
        k[0, at] = (q[0, 0].double() * score / q[0, 0].double().square().sum()).half()
        v[0, at] = rnd(D).half()
    do = rnd(T, 1, D).half()
    kd, vd, dod = k[0, far].double(), v[0, far].double(), do[0, 0].double()
    s = kd @ q[0, 0].double()
    lse = torch.logsumexp(torch.cat([s, torch.tensor([S - 2.0], device=DEV, dtype=torch.float64).log()]), 0)
    p = (s - lse).exp()
    o = (p @ vd).half()
    want = (p * (vd @ dod - (o.double() * dod).sum())) @ kd * sc
    got = _dq(q, k, v, o.view(T, 1, D), lse.float().view(1, T), do, P)
    assert_close(got[0, 0], want, torch.float16, "dq")
