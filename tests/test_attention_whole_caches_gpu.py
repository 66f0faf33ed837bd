"""Gradient caches that a call writes whole, from incoming caches that it leaves alone, against the in-place form on a copy of
them: the same sums in the same order, so the same bits."""
import pytest
import torch

from terapipe_amd import ops

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


# (T, B, H, Dh, P, L, types): slices that end on and off a block of 32 / 64 / 128 keys, caches that end with the slice, within its
# last block and several blocks on; one, two and four waves of 32 keys, the shared form, head dimensions of the first generation
CASES = [(1, 1, 1, 64, 0, 1), (33, 1, 2, 64, 0, 40), (31, 2, 3, 128, 65, 250), (32, 2, 32, 80, 416, 512), (40, 2, 70, 64, 90, 300),
         (64, 1, 40, 128, 64, 257), (300, 1, 24, 96, 11, 400), (16, 2, 4, 16, 37, 131), (70, 1, 3, 32, 60, 300), (130, 2, 130, 64, 0, 131)]


@pytest.mark.parametrize("dtype,gdt", [(torch.float16, torch.float16), (torch.bfloat16, torch.bfloat16),
                                       (torch.float16, torch.float32), (torch.float32, torch.float32)], ids=str)
@pytest.mark.parametrize("T,B,H,Dh,P,L", CASES)
def test_whole_caches_are_the_in_place_ones(dtype, gdt, T, B, H, Dh, P, L):
    g = torch.Generator(device=DEV).manual_seed(T + P)
    BH, E, S = B * H, H * Dh, P + T

    def rnd(*shape, dt=dtype):
        return torch.randn(shape, device=DEV, generator=g).to(dt)
    q, k, v, d_o = rnd(BH, T, Dh), rnd(BH, L, Dh), rnd(BH, L, Dh), rnd(T, B, E)
    ik, iv = rnd(BH, L, Dh, dt=gdt), rnd(BH, L, Dh, dt=gdt)
    o, lse = ops.attn_prefix_fwd(q, k, v, B, H, Dh, T, P, Dh ** -0.5)

    def bwd(gk, gv, flags, **kw):
        dqkv = torch.full((T * B, 3 * E), float("nan"), dtype=dtype, device=DEV)
        ops.attn_prefix_bwd(q, k, v, o, lse, d_o, dqkv, gk, gv, B, H, Dh, T, P, Dh ** -0.5, *flags, **kw)
        return dqkv, gk, gv
    for incoming in (True, False):
        start = (ik, iv) if incoming else (torch.zeros_like(ik), torch.zeros_like(iv))
        want = bwd(start[0].clone(), start[1].clone(), (True,) * 3)
        kept = (ik.clone(), iv.clone())
        fresh = [torch.full_like(ik, float("nan")) for _ in range(2)]
        got = bwd(*fresh, (False,) * 3, whole_caches=True, dk_in=ik if incoming else None, dv_in=iv if incoming else None)
        for a, b, what in zip(got, want, ("dqkv", "dk", "dv")):
            assert torch.equal(a, b), (what, incoming)
        assert torch.equal(ik, kept[0]) and torch.equal(iv, kept[1])
        assert (got[1][:, P:S] == 0).all() and torch.equal(got[2][:, S:], start[1][:, S:])
