"""Losses that see only one of a layer's two cache outputs: the other one's gradient is zero, not both."""
import pytest
import torch


def test_one_incoming_gradient():
    from terapipe_amd.transformer_models import _cache_grads
    cache, g = torch.zeros(2, 3, 8), torch.randn(2, 3, 8)
    for dk, dv in ((g, None), (None, g)):
        gk, gv, k_in, v_in = _cache_grads(cache, dk, dv)
        assert gk.shape == gv.shape == cache.shape
        assert torch.equal(k_in, g if dk is not None else cache) and torch.equal(v_in, g if dv is not None else cache)
    assert _cache_grads(cache, None, None)[2:] == (None, None)
    k_in, v_in = _cache_grads(cache, g, 2 * g)[2:]
    assert torch.equal(k_in, g) and torch.equal(v_in, 2 * g)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16], ids=str)
@pytest.mark.parametrize("attention_only", [False, True])
@pytest.mark.parametrize("side", [0, 1], ids=["k", "v"])
def test_loss_on_one_cache(side, attention_only, dtype):
    import terapipe_amd as ta
    E, H, B, T, P, L = 128, 2, 2, 5, 3, 12
    torch.manual_seed(5)
    layer = ta.ModelParallelTransformerLayer(E, 4 * E, H, device="cuda").to(dtype)
    module = layer.attn if attention_only else layer
    x = torch.randn(T, B, E, device="cuda").to(dtype).requires_grad_()
    start = [torch.randn(B * H, L, E // H, device="cuda").to(dtype) for _ in range(2)]
    g = torch.randn(B * H, L, E // H, device="cuda").to(dtype)

    def run(both):
        ins = [c.clone().requires_grad_() for c in start]
        _, outs = module(x, tuple(ins), P)
        if both:
            grads = [torch.zeros_like(g), torch.zeros_like(g)]
            grads[side] = g
            return torch.autograd.grad(list(outs), [x] + ins + [module.in_proj.weight if attention_only else layer.attn.in_proj.weight], grads)
        return torch.autograd.grad([outs[side]], [x] + ins + [module.in_proj.weight if attention_only else layer.attn.in_proj.weight], [g])
    one, two = run(False), run(True)
    assert all(torch.equal(a, b) for a, b in zip(one, two))
    # the rows that the call does not write keep the gradient of their output, those that it writes hand theirs to x
    dcache = one[1 + side]
    assert torch.equal(dcache[:, :P], g[:, :P]) and torch.equal(dcache[:, P + T:], g[:, P + T:]) and not dcache[:, P:P + T].any()
    assert not one[2 - side].any() and one[0].abs().max() > 0
