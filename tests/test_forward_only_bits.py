"""A forward without gradients gives the bits of the one that autograd sees: activation checkpointing runs the one and differentiates the
other.  Products of a few rows sum in another order only where the caller says that no backward can follow (inference mode)."""
import ctypes

import pytest
import torch
from torch.utils.checkpoint import checkpoint

import oracle
from tests.util import assert_close, load_params_into, make_params

DEV = "cuda"


def test_who_says_that_nothing_is_differentiated(monkeypatch):
    import terapipe_amd as ta
    from terapipe_amd import _layer_core as core
    from terapipe_amd import _lib, ops
    made = []
    monkeypatch.setattr(core, "layers_fwd", lambda images, n, device: made.extend(
        _lib.LayerDesc.from_buffer_copy(images, i * ctypes.sizeof(_lib.LayerDesc)).no_backward for i in range(n)))
    monkeypatch.setattr(ops, "_require_cuda", lambda *tensors: None)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    stack = ta.TransformerLayers(2, 64, 128, 1, dtype=torch.float32, device="cpu")
    x, cache = torch.zeros(4, 1, 64), stack.create_cache(1, 4)
    with torch.no_grad():
        stack(x, cache, 0)
        stack.layers[0](x)
    stack.layers[0](x)
    assert made == [0, 0, 0, 0]
    with torch.inference_mode():
        stack(x, cache, 0)
        stack.layers[0](x)
    assert made[4:] == [1, 1, 1]


def test_no_backward_after_a_forward_that_ruled_it_out():
    from terapipe_amd import _lib
    lib, d = _lib.load(), _lib.LayerBwdDesc()
    f = d.f
    f.dtype, f.T, f.batch, f.heads, f.hidden, f.ffn, f.cache_rows = _lib.TP_F16, 4, 1, 1, 64, 256, 4
    for i in range(12):
        f.w[i] = 4096               # never dereferenced: the call is refused before its first launch
    for names, at in ((_lib.LayerDesc._fields_, f), (_lib.LayerBwdDesc._fields_, d)):
        for name, kind in names:
            if kind is ctypes.c_void_p:
                setattr(at, name, 4096)
    f.no_backward = 1
    assert lib.tp_layer_bwd(ctypes.addressof(d), None, 0, None) == 1 and b"no backward" in lib.tp_last_error()


def _stack(E, F, heads, dtype, activation, n=2):
    import terapipe_amd as ta
    ps = make_params(n, E, F, dtype, seed=E)
    layers = ta.TransformerLayers(n, E, F, heads, dtype=dtype, device=DEV, activation=activation)
    load_params_into(layers, ps, dtype)
    return layers, ps


# up to 8 rows: k splits, tiles of 8 and 16 weight rows, weights beyond 4096 x 4096, a LayerNorm that the product takes itself or not
SIZES = [(2048, 8192, 16, 4, 1, 100), (768, 3072, 12, 2, 1, 5), (640, 2560, 8, 3, 2, 0), (2560, 16384, 32, 8, 1, 3), (5120, 20480, 40, 1, 2, 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("E,F,heads,B,T,P", SIZES, ids=str)
def test_without_gradients_and_checkpointed(E, F, heads, B, T, P, dtype):
    layers, _ = _stack(E, F, heads, dtype, "relu")
    g = torch.Generator(device=DEV).manual_seed(E)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    x, dy = rnd(T, B, E), rnd(T, B, E)
    caches = [rnd(*c.shape) for c in layers.create_cache(B, P + T)]
    run = lambda x, c: layers(x, c, P)[0]
    copies = lambda: [c.clone() for c in caches]
    c0, c1, c2 = copies(), copies(), copies()
    x0, x2 = x.clone().requires_grad_(), x.clone().requires_grad_()
    y0 = run(x0, c0)
    with torch.no_grad():
        y1 = run(x, c1)
    assert torch.equal(y0, y1) and all(torch.equal(a, b) for a, b in zip(c0, c1))
    y2 = checkpoint(lambda x: run(x, c2), x2, use_reentrant=True)
    assert torch.equal(y0, y2)
    y0.backward(dy)
    grads = [p.grad.clone() for p in layers.parameters()]
    layers.zero_grad()
    y2.backward(dy)
    assert torch.equal(x0.grad, x2.grad) and all(torch.equal(a, p.grad) for a, p in zip(grads, layers.parameters()))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("E,F,heads,batch,slices", [
    (128, 512, 2, 1, [1, 3, 8, 1]), (768, 3072, 12, 2, [1, 4, 2]), (640, 2560, 8, 3, [2, 1]), (2560, 16384, 32, 8, [1, 1]),
    (2304, 576, 18, 1, [2, 5, 9]), (2048, 8192, 16, 4, [1, 2])], ids=str)
def test_inference_mode(E, F, heads, batch, slices, dtype):
    layers, ps = _stack(E, F, heads, dtype, "gelu")
    L = sum(slices)
    g = torch.Generator().manual_seed(L)
    x, dy = (torch.randn(L, batch, E, generator=g).to(dtype) for _ in range(2))
    leaf = [{k: v.clone().requires_grad_(True) for k, v in p.items()} for p in ps]
    want, _, _ = oracle.terapipe_forward_backward(leaf, x.float(), dy.float(), heads, [batch], slices, activation="gelu")
    with torch.inference_mode():
        cache, single, done, out = layers.create_cache(batch, L), layers.create_cache(batch, L), 0, []
        for n in slices:
            y, cache = layers(x[done:done + n].to(DEV), cache, done)
            z = x[done:done + n].to(DEV)
            for i, layer in enumerate(layers.layers):
                z, _ = layer(z, (single[2 * i], single[2 * i + 1]), done)
            assert torch.equal(y, z)        # the stack gives its layers' bits
            out.append(y)
            done += n
    assert all(torch.equal(a, b) for a, b in zip(cache, single))
    assert_close(torch.cat(out), want, dtype, "y")
