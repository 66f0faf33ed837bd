"""A stack without gradients calls its layers one by one wherever somebody could see that it does not (CPU: the library
calls are replaced by a note of who asked for them)."""
import pytest
import torch


@pytest.fixture
def stack(monkeypatch):
    """(layers, inputs, calls): calls lists the number of layers of every library call."""
    import terapipe_amd as ta
    from terapipe_amd import _layer_core as core
    calls = []

    def stack_forward_only(layers, x, caches, cache_len):
        calls.append(len(layers))
        return x + len(layers)

    monkeypatch.setattr(core, "stack_forward_only", stack_forward_only)
    layers = ta.TransformerLayers(3, 64, 128, 1, dtype=torch.float32, device="cpu")
    x, cache = torch.zeros(2, 1, 64), layers.create_cache(1, 4)

    def run():
        calls.clear()
        with torch.no_grad():
            y, out = layers(x, cache, 1)
        assert (y == 3).all() and [c.data_ptr() for c in out] == [c.data_ptr() for c in cache]
        return calls

    return layers, run


def test_plain_layers_are_one_call(stack):
    layers, run = stack
    assert run() == [3]
    layers.layers.append(layers.layers[0])      # n_layers of them, as with gradients
    assert run() == [3]


@pytest.mark.parametrize("pre", [False, True])
def test_forward_hooks(stack, pre):
    layers, run = stack
    seen = []
    register = layers.layers[1].register_forward_pre_hook if pre else layers.layers[1].register_forward_hook
    handle = register(lambda *a: seen.append(a[0]))
    assert run() == [1, 1, 1] and seen == [layers.layers[1]]
    handle.remove()
    assert run() == [3]
    g = torch.nn.modules.module
    handle = (g.register_module_forward_pre_hook if pre else g.register_module_forward_hook)(lambda *a: seen.append(a[0]))
    try:
        assert run() == [1, 1, 1] and list(layers.layers) == [m for m in seen[1:] if m in list(layers.layers)]
    finally:
        handle.remove()


def test_other_forwards(stack):
    import terapipe_amd as ta
    layers, run = stack
    plain = layers.layers[1]
    seen = []

    class Noted(ta.ModelParallelTransformerLayer):
        def forward(self, *a):
            seen.append("subclass")
            return super().forward(*a)

    class Wrapper(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        def forward(self, *a):
            seen.append("wrapper")
            return self.inner(*a)

    for other, word in ((Noted(64, 128, 1), "subclass"), (Wrapper(plain), "wrapper")):
        layers.layers[1] = other
        assert run() == [1, 1, 1] and seen.pop() == word
    layers.layers[1] = plain
    inner = plain.forward
    plain.forward = lambda *a: seen.append("instance") or inner(*a)       # as offloading libraries do
    assert run() == [1, 1, 1] and seen == ["instance"]
    del plain.forward
    assert run() == [3]


def test_traces_and_forward_mode_see_the_autograd_function(stack, monkeypatch):
    """What follows a computation without gradients meets the layer as the node it is with gradients."""
    from terapipe_amd import transformer_models as tm
    layers, run = stack
    seen = []

    class Node:
        @staticmethod
        def apply(heads, cache_len, activation, opts, x, k, v, *params):
            seen.append("node")
            return (x + 1, k, v)

    monkeypatch.setattr(tm, "_LayerFunction", Node)
    assert run() == [3] and not seen
    with torch.autograd.forward_ad.dual_level():
        assert run() == [] and len(seen) == 3
    seen.clear()
    monkeypatch.setattr(torch._C, "_get_tracing_state", lambda: object())
    assert run() == [] and len(seen) == 3
