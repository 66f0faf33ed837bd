"""Deferred weight gradients: a slice is deferred or not as its forward found the switch, and what its weight gradients read
is what its forward wrote (CPU: the library calls are replaced by a look at their descriptors)."""
import pytest
import torch

from terapipe_amd import _layer_core as core
from terapipe_amd import _lib, ops

INPUTS = ("xn", "o", "hn", "a")


@pytest.fixture
def descriptors(monkeypatch):
    """[(forward or backward, descriptor)] of the layer calls made."""
    made = []

    def forward(images, n, device):
        made.append(("forward", _lib.LayerDesc.from_buffer_copy(images)))

    def backward(image, device):
        made.append(("backward", _lib.LayerBwdDesc.from_buffer_copy(image)))

    monkeypatch.setattr(core, "layers_fwd", forward)
    monkeypatch.setattr(core, "layer_bwd_native", backward)
    monkeypatch.setattr(ops, "_require_cuda", lambda *tensors: None)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    return made


def _slice(layer, T=4, L=8, P=0, cache=None):
    cache = cache or tuple(torch.zeros(1, L, 64) for _ in range(2))
    y, out = layer(torch.zeros(T, 1, 64, requires_grad=True), tuple(c.detach().requires_grad_() for c in cache), P)
    return y, out, cache


@pytest.mark.parametrize("before", [False, True])
def test_the_switch_changes_between_forward_and_backward(descriptors, before):
    import terapipe_amd as ta
    layer = ta.ModelParallelTransformerLayer(64, 128, 1)
    layer.defer_weight_grads = before
    y, _, _ = _slice(layer)
    layer.defer_weight_grads = not before
    _slice(layer)
    y.sum().backward()
    (_, f), _, (_, b) = descriptors
    assert b.wg_rows == 4 and [getattr(b, "wg_" + n) for n in INPUTS] == [getattr(f, n) for n in INPUTS]
    assert all(p.grad is not None for p in layer.parameters())


def test_two_slices(descriptors):
    """The weight gradients go out once, over both slices' rows, which lie one after the other."""
    import terapipe_amd as ta
    layer = ta.ModelParallelTransformerLayer(64, 128, 1)
    layer.defer_weight_grads = True
    y0, _, cache = _slice(layer)
    y1, _, _ = _slice(layer, P=4, cache=cache)
    y1.sum().backward()
    y0.sum().backward()
    (_, f0), (_, f1), (_, b1), (_, b0) = descriptors
    assert b1.wg_rows == 0 and b0.wg_rows == 8
    for n, width in zip(INPUTS, (64, 64, 64, 128)):
        assert getattr(b0, "wg_" + n) == getattr(f0, n) and getattr(f1, n) == getattr(f0, n) + 4 * width * 4


def test_the_linears_inputs_are_kept_once(descriptors):
    """By the slice, or by the sequence with deferred weight gradients: not by both."""
    import terapipe_amd as ta
    layer = ta.ModelParallelTransformerLayer(64, 128, 1)
    sizes = {}
    for layer.defer_weight_grads in (False, True):
        y, _, _ = _slice(layer, T=32, L=64)
        sizes[layer.defer_weight_grads] = y.grad_fn.kept[3].numel()
    assert sizes[False] - sizes[True] == 32 * (3 * 64 + 128) * 4
