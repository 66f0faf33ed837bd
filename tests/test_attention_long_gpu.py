"""The attention kernels for whole sequences and long slices (workgroups of 128 queries) forced at their edges against fp32:
rows, blocks and key tiles that end inside a workgroup's, prefixes of every alignment, references that move on most tiles."""
import ctypes

import pytest
import torch

from tests.util import assert_close

DEV = "cuda"


def _reference(q, k, v, P):
    """o and log-sum-exp in fp32, [B*H, T, Dh]."""
    T, S = q.shape[1], k.shape[1]
    s = torch.bmm(q.float(), k.float().transpose(1, 2).contiguous())
    mask = torch.arange(S, device=q.device)[None] > P + torch.arange(T, device=q.device)[:, None]
    s.masked_fill_(mask, float("-inf"))
    return torch.bmm(torch.softmax(s, -1), v.float()), torch.logsumexp(s, -1)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("D", [64, 80, 96, 128])
@pytest.mark.parametrize("B,H,T,P,drift", [(1, 3, 1, 0, 0.0), (2, 1, 33, 95, 0.0), (1, 2, 128, 0, 0.0), (1, 2, 129, 1, 0.0),
                                           (2, 3, 300, 0, 0.0), (1, 5, 130, 500, 0.0), (1, 1, 256, 255, 6.0), (1, 2, 384, 37, -6.0)],
                         ids=str)
def test_forward(B, H, T, P, drift, D, dtype):
    from terapipe_amd import ops
    S = P + T
    g = torch.Generator(device=DEV).manual_seed(T + 7 * P + D)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    # drift: scores that grow (or fall) along the keys by several kSlack
    q, k = rnd(B * H, T, D) * D ** -0.5, rnd(B * H, S + 3, D)
    if drift:
        q[:, :, 0], k[:, :S, 0] = 1.0, drift * 5.0 * torch.linspace(0, 1, S, device=DEV)
    q, k, v = q.to(dtype), k.to(dtype), rnd(B * H, S + 3, D).to(dtype)
    k[:, S:], v[:, S:] = float("nan"), float("nan")       # rows past the slice are never used
    o, lse = ops.attn_prefix_fwd(q, k, v, batch=B, heads=H, head_dim=D, T=T, cache_len=P, q_scale=D ** -0.5, variant=32)
    want, want_lse = _reference(q, k[:, :S], v[:, :S], P)
    assert_close(o, want.view(B, H, T, D).permute(2, 0, 1, 3).reshape(T, B, H * D), dtype, "o")
    assert_close(lse, want_lse, torch.float32, "lse")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("B,H,D,T,P,acc,incoming,zero", [
    (2, 128, 64, 129, 0, 0, 0, 0), (1, 256, 64, 130, 67, 1, 1, 1), (4, 48, 80, 128, 1, 0, 1, 0), (1, 110, 96, 200, 131, 1, 0, 1),
    (2, 56, 128, 193, 63, 1, 1, 0), (1, 96, 128, 255, 0, 0, 0, 0),
    (1, 3, 96, 1, 70, 1, 1, 1), (2, 2, 128, 33, 95, 0, 1, 0), (1, 2, 64, 40, 0, 0, 0, 0),
    (1, 257, 80, 1, 0, 0, 0, 0), (1, 300, 96, 7, 25, 1, 1, 1), (1, 384, 128, 16, 48, 1, 0, 1)], ids=str)
def test_backward(B, H, D, T, P, acc, incoming, zero, dtype):
    """Both backward forms: with gradient caches, and dQ with the one-pass dK / dV (the last rows: the first of them alone, for which
    few workgroups are enough)."""
    from terapipe_amd import ops
    S, BH, sc = P + T, B * H, D ** -0.5
    g = torch.Generator(device=DEV).manual_seed(T + 7 * P + D)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    q, k, v, do = (rnd(BH, S, D) * sc).to(dtype), rnd(BH, S + 3, D).to(dtype), rnd(BH, S + 3, D).to(dtype), rnd(S, B, H * D).to(dtype)
    k[:, S:], v[:, S:] = float("nan"), float("nan")       # rows past the slice are never used
    gk, gv = rnd(BH, S + 3, D).to(dtype), rnd(BH, S + 3, D).to(dtype)
    gk0, gv0 = gk.double()[:, :S], gv.double()[:, :S]

    def reference(first, keys):     # queries [first, S) against the keys [0, keys): dq, dk, dv, o, lse in fp64
        qd, kd, vd = (t.double().requires_grad_() for t in (q[:, first:], k[:, :keys], v[:, :keys]))
        s = torch.bmm(qd, kd.transpose(1, 2).contiguous())
        s = s.masked_fill(torch.arange(keys, device=DEV)[None] > torch.arange(first, S, device=DEV)[:, None], float("-inf"))
        od = torch.bmm(torch.softmax(s, -1), vd)
        od.backward(do[first:].double().view(S - first, B, H, D).permute(1, 2, 0, 3).reshape(BH, S - first, D))
        return qd.grad, kd.grad, vd.grad, od.detach(), torch.logsumexp(s, -1).detach()

    rows = lambda t: t.reshape(B, H, -1, D).permute(2, 0, 1, 3).reshape(-1, H, D)
    # the slice [P, S) with gradient caches
    dq, dk, dv, o, lse = reference(P, S)
    o16, lse32 = rows(o).reshape(T, B, H * D).to(dtype), lse.float()
    dqkv = torch.full((T * B, 3 * H * D), float("nan"), device=DEV, dtype=dtype)
    ops.attn_prefix_bwd(q[:, P:].contiguous(), k, v, o16, lse32, do[P:].contiguous(), dqkv, gk, gv, B, H, D, T, P, sc,
                        bool(acc), bool(incoming), bool(zero))
    part = dqkv.view(T * B, H, 3, D)
    assert_close(part[:, :, 0], rows(dq * sc), dtype, "dq")
    for i, (got, want, old) in enumerate(((gk, dk, gk0), (gv, dv, gv0)), 1):
        assert_close(part[:, :, i], rows(want[:, P:] + (old[:, P:] if incoming else 0)), dtype, "dk dv"[3 * i - 3:3 * i - 1])
        if P:
            assert_close(got[:, :P], want[:, :P] + (old[:, :P] if acc else 0), dtype, "prefix")
        assert torch.equal(got[:, P:S].double(), torch.zeros_like(old[:, P:]) if zero else old[:, P:])
    # the first T positions, their keys against every query of [0, S)
    dq, dk, dv, o, lse = reference(0, S)
    delta = (o * do.double().view(S, B, H, D).permute(1, 2, 0, 3).reshape(BH, S, D)).sum(-1).float()
    dqkv.fill_(float("nan"))
    ops.attn_suffix_dkdv(k, v, q, do, lse.float(), delta, dqkv, B, H, D, 0, T, S)
    part = dqkv.view(T * B, H, 3, D)
    assert_close(part[:, :, 1], rows(dk[:, :T]), dtype, "suffix dk")
    assert_close(part[:, :, 2], rows(dv[:, :T]), dtype, "suffix dv")
    assert part[:, :, 0].isnan().all()


# (B * H, head dim, T, P) -> whether the gradient-cache dK / dV takes the shared form
@pytest.mark.parametrize("pairs,D,T,P,want", [
    (256, 128, 1, 0, 1), (257, 80, 1, 0, 0), (511, 96, 32, 0, 0), (512, 128, 1, 31, 1), (257, 128, 33, 0, 1), (384, 80, 16, 48, 0),
    (385, 80, 16, 48, 1), (384, 96, 17, 47, 1), (384, 128, 16, 49, 1), (768, 128, 1, 0, 1), (40, 128, 256, 768, 1), (300, 64, 8, 8, 0)], ids=str)
def test_short_calls_of_a_second_round_keep_the_form_with_a_wave_per_key_block(pairs, D, T, P, want):
    from terapipe_amd import _lib as L
    d = L.AttnDesc()
    d.dtype = d.grad_cache_dtype = L.TP_F16
    d.batch, d.heads, d.head_dim, d.T, d.cache_len, d.cache_rows = 1, pairs, D, T, P, T + P
    for name in ("q", "k_cache", "v_cache", "o", "lse", "d_o", "delta", "dqkv", "dk_cache", "dv_cache"):
        setattr(d, name, 4096)
    keys = ctypes.c_int(-1)
    assert L.load().tp_attn_bwd_forms(ctypes.byref(d), None, ctypes.byref(keys)) == 0
    assert keys.value == want


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("D", [64, 80, 96, 128])
@pytest.mark.parametrize("B,H,T,P", [(1, 3, 1, 0), (2, 1, 63, 2), (1, 2, 64, 31), (1, 2, 65, 95), (1, 1, 193, 500), (3, 13, 128, 0), (2, 300, 33, 5),
                                     (1, 520, 65, 0), (2, 260, 97, 70)], ids=str)
def test_dq(B, H, T, P, D, dtype):
    """Blocks of 64 and (the last three) of 128 queries: those that end inside a block, key tiles that end inside or that only one of
    two waves sees, fewer tiles than the rings have slots; 39 pairs of two blocks go in the paired order of one round."""
    from terapipe_amd import _lib as L
    from terapipe_amd import ops
    S, BH, sc = P + T, B * H, D ** -0.5
    g = torch.Generator(device=DEV).manual_seed(T + 7 * P + D)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    q, k, v, do = (rnd(BH, T, D) * sc).to(dtype), rnd(BH, S + 3, D).to(dtype), rnd(BH, S + 3, D).to(dtype), rnd(T, B, H * D).to(dtype)
    k[:, S:], v[:, S:] = float("nan"), float("nan")       # rows past the slice are never used
    qd, kd, vd = (t.double() for t in (q, k[:, :S].contiguous(), v[:, :S].contiguous()))
    s = torch.bmm(qd, kd.transpose(1, 2).contiguous())
    s = s.masked_fill(torch.arange(S, device=DEV)[None] > P + torch.arange(T, device=DEV)[:, None], float("-inf"))
    p, o, lse = torch.softmax(s, -1), torch.bmm(torch.softmax(s, -1), vd), torch.logsumexp(s, -1)
    dod = do.double().view(T, B, H, D).permute(1, 2, 0, 3).reshape(BH, T, D)
    delta = (o * dod).sum(-1)
    want = torch.bmm(p * (torch.bmm(dod, vd.transpose(1, 2).contiguous()) - delta[..., None]), kd) * sc
    o16 = o.view(B, H, T, D).permute(2, 0, 1, 3).reshape(T, B, H * D).to(dtype).contiguous()
    got_delta, lse32 = torch.full((BH, T), float("nan"), device=DEV), lse.float()
    dqkv = torch.full((T * B, 3 * H * D), float("nan"), device=DEV, dtype=dtype)
    d = ops._attn_desc(q, k, v, o16, lse32, B, H, D, T, P, sc)
    d.dq_only, d.reserved2, d.grad_cache_dtype = 1, 32, d.dtype
    d.d_o, d.delta, d.dqkv = do.data_ptr(), got_delta.data_ptr(), dqkv.data_ptr()
    L.check(L.load().tp_attn_prefix_bwd(ctypes.byref(d), None, 0, ops._stream()), "tp_attn_prefix_bwd")
    part = dqkv.view(T * B, H, 3, D)
    assert_close(part[:, :, 0], want.view(B, H, T, D).permute(2, 0, 1, 3).reshape(-1, H, D), dtype, "dq")
    assert part[:, :, 1:].isnan().all()
    rounded = (o16.double().view(T, B, H, D).permute(1, 2, 0, 3).reshape(BH, T, D) * dod).sum(-1)
    assert_close(got_delta, rounded, torch.float32, "delta")


@pytest.mark.parametrize("pairs,D,T,P,want", [
    (160, 128, 64, 0, 1), (159, 128, 64, 0, 0), (400, 128, 63, 0, 0), (40, 80, 256, 768, 1), (8, 96, 1280, 0, 0), (16, 128, 640, 1400, 1),
    (10, 128, 2048, 0, 1), (256, 64, 64, 0, 1), (255, 64, 64, 0, 0), (16, 64, 2048, 0, 1), (8, 64, 2048, 0, 0)], ids=str)
def test_who_shares_the_tiles_of_dq(pairs, D, T, P, want):
    from terapipe_amd import _lib as L
    d = L.AttnDesc()
    d.dtype = d.grad_cache_dtype = L.TP_F16
    d.batch, d.heads, d.head_dim, d.T, d.cache_len, d.cache_rows = 1, pairs, D, T, P, T + P
    for name in ("q", "k_cache", "v_cache", "o", "lse", "d_o", "delta", "dqkv", "dk_cache", "dv_cache"):
        setattr(d, name, 4096)
    queries = ctypes.c_int(-1)
    assert L.load().tp_attn_bwd_forms(ctypes.byref(d), ctypes.byref(queries), None) == 0
    assert queries.value == want
