"""What a layer's kernels are handed: strides of the parameters."""
import pytest
import torch

from tests.util import assert_close


def _layer(E, H, F, dtype, activation="gelu", seed=3, device="cuda"):
    import terapipe_amd as ta
    torch.manual_seed(seed)
    layer = ta.ModelParallelTransformerLayer(E, F, H, device=device, activation=activation).to(dtype)
    with torch.no_grad():
        for p in layer.parameters():
            p.add_(torch.randn_like(p) * 0.02)
    return layer


def _replace_weights(layer, change):
    for m in (layer.attn.in_proj, layer.attn.out_proj, layer.fc1, layer.fc2):
        m.weight = torch.nn.Parameter(change(m.weight.detach()))


def _column_range(w, before=8, after=16):
    """w as columns [before, before + K) of a wider matrix of other values."""
    wide = torch.full((w.shape[0], before + w.shape[1] + after), 7.0, dtype=w.dtype, device=w.device)
    wide[:, before:before + w.shape[1]] = w
    return wide[:, before:before + w.shape[1]]


def _forward_backward(layer, x, dy, P=3):
    B, L = x.shape[1], P + x.shape[0]
    H, Dh = layer.attn.num_heads, layer.attn.head_dim
    g = torch.Generator(device="cuda").manual_seed(1)
    caches = [torch.randn(B * H, L, Dh, generator=g, device="cuda").to(x.dtype).requires_grad_() for _ in range(2)]
    x = x.clone().requires_grad_()
    y, _ = layer(x, tuple(caches), P)
    y.backward(dy)
    with torch.no_grad():
        y0, _ = layer(x, tuple(c.detach() for c in caches), P)
    return [y.detach(), y0, x.grad] + [c.grad for c in caches] + [p.grad for p in layer.param_list()]


def test_addresses_and_row_pitches(monkeypatch):
    from terapipe_amd import _layer_core as core
    from terapipe_amd import _lib, ops
    monkeypatch.setattr(ops, "_require_cuda", lambda *tensors: None)
    layer = _layer(64, 1, 128, torch.float16, device="cpu")
    ptrs, ldw = core.operands(layer.param_list(), torch.float16)
    assert ptrs == [p.data_ptr() for p in layer.param_list()] and list(ldw) == [0] * 4
    _replace_weights(layer, _column_range)
    ptrs, ldw = core.operands(layer.param_list(), torch.float16)
    assert ptrs == [p.data_ptr() for p in layer.param_list()] and ldw == [64 + 24] * 3 + [128 + 24]
    for change in (lambda w: w.t().contiguous().t(), lambda w: w[:1].expand(w.shape), lambda w: torch.cat([w, w], 1)[:, ::2]):
        _replace_weights(layer, change)
        with pytest.raises(_lib.TeraPipeHipError, match="in_proj.weight: strides"):
            core.operands(layer.param_list(), torch.float16)
    layer = _layer(64, 1, 128, torch.float16, device="cpu")
    layer.fc1.bias = torch.nn.Parameter(torch.zeros(256, dtype=torch.float16)[::2])
    with pytest.raises(_lib.TeraPipeHipError, match="fc1.bias: strides"):
        core.operands(layer.param_list(), torch.float16)


@pytest.mark.gpu
@pytest.mark.parametrize("T,dtype", [(5, torch.float16), (70, torch.bfloat16), (9, torch.float32)], ids=str)
def test_weights_that_are_column_ranges(T, dtype):
    """The same bits as from dense weights, with and without gradients (the sums over rows of the vector parameters'
    gradients are atomic: their order is not fixed)."""
    x, dy = (torch.randn(T, 2, 128, device="cuda").to(dtype) for _ in range(2))
    layer = _layer(128, 2, 512, dtype)
    ref = _forward_backward(layer, x, dy)
    _replace_weights(layer, _column_range)
    layer.zero_grad()
    got = _forward_backward(layer, x, dy)
    for i, (a, b) in enumerate(zip(got, ref)):
        if a.dim() > 1:
            assert torch.equal(a, b), "tensor %d" % i
        else:
            assert_close(a, b, dtype, "tensor %d" % i, 1.0 if dtype == torch.float32 else 0.1)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32], ids=str)
def test_forward_only_stack_of_unequal_layers(dtype):
    """FFN width, heads and activation are each layer's own, also where no gradients are asked for."""
    import terapipe_amd as ta
    E, T, B, P = 256, 6, 2, 5
    layers = ta.TransformerLayers(4, E, 4 * E, 4, dtype=dtype, device="cuda")
    shapes = [(4, 4 * E, "relu"), (2, 2 * E, "gelu"), (4, 6 * E, "gelu"), (4, E, "relu")]
    for i, (H, F, activation) in enumerate(shapes):
        layers.layers[i] = _layer(E, H, F, dtype, activation, seed=i)
    x = torch.randn(T, B, E, device="cuda").to(dtype)
    caches = [torch.randn(c.shape, device="cuda").to(dtype) for c in layers.create_cache(B, P + T)]
    ref, _ = layers(x, [c.clone().requires_grad_() for c in caches], P)
    with torch.no_grad():
        got, _ = layers(x, caches, P)
    assert_close(got, ref, dtype, "y", 1.0 if dtype == torch.float32 else 0.1)


@pytest.mark.gpu
@pytest.mark.parametrize("grad", [False, True])
def test_host_memory_and_other_types_are_refused(grad):
    """Nothing is launched: parameters or caches in host memory, and parameters of another type than the input."""
    from terapipe_amd import _lib
    layer = _layer(128, 2, 512, torch.float16)
    x = torch.randn(3, 1, 128, device="cuda").half()
    caches = [torch.zeros(2, 4, 64, dtype=torch.float16, device="cuda") for _ in range(2)]
    with torch.set_grad_enabled(grad):
        layer(x, tuple(caches), 0)
        for i in range(2):
            with pytest.raises(_lib.TeraPipeHipError, match="no CPU path"):
                layer(x, tuple(c.cpu() if i == j else c for j, c in enumerate(caches)), 0)
        with pytest.raises(_lib.TeraPipeHipError, match="no CPU path"):
            layer(x.cpu(), tuple(caches), 0)
        for name in ("fc1.weight", "fc_ln.bias"):
            module = getattr(layer, name.split(".")[0])
            kept = getattr(module, name.split(".")[1])
            for other, message in ((kept.detach().cpu(), "no CPU path"), (kept.detach().float(), name + " is torch.float32")):
                setattr(module, name.split(".")[1], torch.nn.Parameter(other))
                with pytest.raises(_lib.TeraPipeHipError, match=message):
                    layer(x, tuple(caches), 0)
            setattr(module, name.split(".")[1], kept)


def test_a_layer_can_be_copied_and_pickled():
    import copy
    import io
    layer = _layer(64, 1, 128, torch.float16, device="cpu")
    layer._grad_options.pending[7] = object()
    f = io.BytesIO()
    torch.save(layer, f)
    f.seek(0)
    for other in (copy.deepcopy(layer), torch.load(f, weights_only=False)):
        assert all(torch.equal(a, b) for a, b in zip(other.param_list(), layer.param_list()))
        assert not other._grad_options.pending and not other._grad_options.inputs
        assert other._grad_options is not layer._grad_options


def test_the_backward_reads_the_parameters_where_they_are_then(monkeypatch):
    """Not where they were when the forward ran: storage that was replaced in between may be anybody's."""
    from terapipe_amd import _layer_core as core
    from terapipe_amd import _lib, ops
    made = []
    monkeypatch.setattr(core, "layers_fwd", lambda images, n, device: made.append(_lib.LayerDesc.from_buffer_copy(images)))
    monkeypatch.setattr(core, "layer_bwd_native", lambda image, device: made.append(_lib.LayerBwdDesc.from_buffer_copy(image).f))
    monkeypatch.setattr(ops, "_require_cuda", lambda *tensors: None)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    layer = _layer(64, 1, 128, torch.float32, device="cpu")
    y, _ = layer(torch.zeros(4, 1, 64, requires_grad=True))
    kept = [p.data for p in layer.param_list()]         # (keeps the old memory from being handed out again)
    for p in layer.param_list():
        p.data = _column_range(p.data) if p.dim() == 2 else p.data.clone()
    y.sum().backward()
    forward, backward = made
    assert list(forward.w) == [t.data_ptr() for t in kept] and list(forward.ldw) == [0] * 4
    assert list(backward.w) == [p.data_ptr() for p in layer.param_list()] and list(backward.ldw) == [64 + 24] * 3 + [128 + 24]
    same = [name for name, _ in _lib.LayerDesc._fields_ if name not in ("w", "ldw")]
    assert [getattr(forward, n) for n in same] == [getattr(backward, n) for n in same]


@pytest.mark.gpu
def test_parameters_that_move_between_forward_and_backward():
    layer = _layer(128, 2, 512, torch.float16)
    x, dy = (torch.randn(9, 2, 128, device="cuda").half() for _ in range(2))
    ref = _forward_backward(layer, x, dy)[5:]
    layer.zero_grad()
    g = torch.Generator(device="cuda").manual_seed(1)
    caches = [torch.randn(4, 12, 64, generator=g, device="cuda").half().requires_grad_() for _ in range(2)]
    y, _ = layer(x.clone().requires_grad_(), tuple(caches), 3)
    for p in layer.param_list():
        old, p.data = p.data, p.data.clone()
        old.fill_(float("nan"))
    del old
    junk = [torch.full((128, 512), float("nan"), dtype=torch.float16, device="cuda") for _ in range(8)]
    y.backward(dy)
    for i, (p, r) in enumerate(zip(layer.param_list(), ref)):
        assert_close(p.grad, r, torch.float16, "parameter %d" % i, 0.1)
    assert all(t.isnan().all() for t in junk)
