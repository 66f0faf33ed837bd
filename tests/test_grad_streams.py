"""Which gradients the kernels add to .grad themselves: the rule on the CPU, and layers whose slices run on several streams."""
import pytest
import torch

from tests.util import assert_close


class _Twice(torch.autograd.Function):
    """y = 2 x p; its backward asks whether it may add to p.grad and does so if it may."""

    @staticmethod
    def forward(ctx, x, p, stream, log):
        ctx.save_for_backward(x)
        ctx.p, ctx.stream, ctx.log = p, stream, log
        return 2 * x * p

    @staticmethod
    def backward(ctx, dy):
        from terapipe_amd import _autograd, ops
        (x,) = ctx.saved_tensors
        ops._stream.now = ctx.stream
        ours = _autograd.engine_adds_to_grad(ctx, (ctx.p,), 1)
        ctx.log.append(ours)
        if ours:
            ctx.p.grad = (0 if ctx.p.grad is None else ctx.p.grad) + (2 * x * dy).detach()
            return None, None, None, None
        return None, 2 * x * dy, None, None


def _twice(x, p, stream=0, log=None):
    """As the layers call theirs, on a stream."""
    from terapipe_amd import _autograd, ops
    ops._stream.now = stream
    fresh = _autograd.fresh_leaves([p])
    y = _Twice.apply(x, p, stream, log)
    _autograd.note_leaves(y.grad_fn, 1, fresh)
    return y


@pytest.fixture
def streams(monkeypatch):
    from terapipe_amd import ops

    def current():
        return current.now

    current.now = 0
    monkeypatch.setattr(ops, "_stream", current)
    return current


def _slices(p, streams_of, log):
    return [_twice(torch.full((3,), float(i + 1)), p, s, log).sum() for i, s in enumerate(streams_of)]


def test_only_on_the_stream_of_the_engines_own_addition(streams):
    """The AccumulateGrad node is the first forward's: slices on its stream add, others hand their gradients over."""
    for on in ([0, 0, 0], [7, 7, 7], [7, 0, 7], [0, 7, 9]):
        p, log = torch.nn.Parameter(torch.ones(3)), []
        for y in _slices(p, on, log):
            y.backward()
        assert log == [s == on[0] for s in on]
        assert torch.equal(p.grad, torch.full((3,), 12.0))


def test_a_node_that_somebody_else_made(streams):
    """By using the parameter first, by holding its node; a parameter that is used again by nobody is ours again."""
    p, log = torch.nn.Parameter(torch.ones(3)), []
    other = (p * 0.5).sum()
    for y in _slices(p, [0, 0], log) + [other]:
        y.backward()
    assert log == [False, False] and torch.equal(p.grad, torch.full((3,), 6.5))
    node = torch.autograd.graph.get_gradient_edge(p).node
    _slices(p, [0], log)[0].backward()
    assert log.pop() is False and node.variable is p
    del node, other, y
    _slices(p, [0], log)[0].backward()
    assert log.pop() is True and torch.equal(p.grad, torch.full((3,), 10.5))


def test_two_threads_make_the_node_at_once(streams):
    """Both found no node and both note their own stream: neither is believed."""
    from terapipe_amd import _autograd
    p, log = torch.nn.Parameter(torch.ones(3)), []
    y0, y1 = _twice(torch.ones(3), p, 0, log), _twice(torch.ones(3), p, 5, log)
    _autograd.note_leaves(y1.grad_fn, 1, [0])
    y0.sum().backward()
    y1.sum().backward()
    assert log == [False, False]


def test_who_looks_at_gradients(streams):
    """Hooks on the parameter or on its node, torch.autograd.grad and a graph of the backward get tensors; hooks that are
    gone, or on something else, do not count."""
    p, log = torch.nn.Parameter(torch.ones(3)), []
    outs = _slices(p, [0] * 9, log)
    node = outs[0].grad_fn.next_functions[0][0].next_functions[1][0]
    one = torch.full((3,), 1.0)
    outs[0].backward()
    seen = []
    for i, register in ((1, lambda: p.register_hook(seen.append)), (2, lambda: node.register_prehook(lambda g: seen.append(g[0]))),
                        (3, lambda: node.register_hook(lambda _, g: seen.append(g[0]))),
                        (4, lambda: p.register_post_accumulate_grad_hook(lambda q: seen.append(q.grad - before)))):
        before = p.grad.clone()
        handle = register()
        outs[i].backward()
        handle.remove()
        assert torch.equal(seen.pop(), 2 * (i + 1) * one) and not seen
    assert log == [True] + [False] * 4 and torch.equal(p.grad, 30 * one)
    assert torch.equal(torch.autograd.grad(outs[5], p)[0], 12 * one)
    elsewhere = torch.nn.Linear(1, 1).register_forward_hook(print)
    torch.autograd.backward([outs[6]], inputs=[p])
    elsewhere.remove()
    outs[7].backward(create_graph=True)
    outs[8].backward()
    assert log[5:] == [False, True, False, True] and torch.equal(p.grad.detach(), (30 + 14 + 16 + 18) * one)


def test_parameters_that_are_no_leaves_or_frozen(streams):
    p, log = torch.nn.Parameter(torch.ones(3)), []
    for q in (p * 1, torch.ones(3)):
        for _ in range(2):
            x = torch.ones(3, requires_grad=True)
            (_twice(x, q, 0, log) + x).sum().backward(retain_graph=True)
    assert log == [False] * 4


@pytest.mark.parametrize("grad", [None, "float64", "strided", "shape", "sparse", "offset"])
def test_gradients_the_kernels_cannot_write(grad):
    import terapipe_amd as ta
    from terapipe_amd import transformer_models as tm
    w = ta.ModelParallelTransformerLayer(64, 128, 1).param_dict()
    for p in w.values():
        p.grad = torch.zeros_like(p)
    assert tm._grads_can_go_in_place(w)
    p = w["fc1.weight"]
    p.grad = None
    if grad == "float64":
        p.grad_dtype = None
    other = {"float64": lambda: torch.zeros_like(p, dtype=torch.float64), "strided": lambda: torch.zeros(64, 128).t(),
             "sparse": lambda: torch.zeros_like(p).to_sparse(), "offset": lambda: torch.zeros(128 * 64 + 1)[1:].view(128, 64)}
    if grad in other:
        p.grad = other[grad]()
    elif grad == "shape":
        w["fc1.weight"] = p = torch.nn.Parameter(p.detach()[:, :32].contiguous())
        p.grad = torch.zeros_like(p)
        p.data = torch.zeros(128, 64)
    assert not tm._grads_can_go_in_place(w)


class _Slow(torch.autograd.Function):
    """Identity whose backward keeps its stream busy first."""

    @staticmethod
    def forward(ctx, x):
        return x.view_as(x)

    @staticmethod
    def backward(ctx, dy):
        torch.cuda._sleep(20_000_000)
        return dy


@pytest.mark.gpu
@pytest.mark.parametrize("foreign", [False, True])
@pytest.mark.parametrize("n_streams", [0, 1, 2, 3])
def test_slices_on_several_streams(n_streams, foreign, monkeypatch):
    """The forwards of four inputs on other streams than the backward's caller, .grad there already: complete sums as soon as
    the calling stream looks.  One stream (its own or the caller's): the kernels add from the second backward on.  foreign:
    the weight is used by somebody else first, on a stream of theirs."""
    import terapipe_amd as ta
    from terapipe_amd import _layer_core as core
    from terapipe_amd import _lib
    torch.manual_seed(3)
    layer = ta.ModelParallelTransformerLayer(256, 1024, 4, device="cuda", activation="gelu").half()
    params = layer.param_list()
    xs, dy = [torch.randn(32, 2, 256, device="cuda").half() for _ in range(4)], torch.randn(32, 2, 256, device="cuda").half()
    refs = [torch.autograd.grad(layer(x)[0], params, dy) for x in xs]
    added = []
    native = core.layer_bwd_native

    def noted(image, device):
        added.append(_lib.LayerBwdDesc.from_buffer(image).wg_accumulate)
        native(image, device)

    monkeypatch.setattr(core, "layer_bwd_native", noted)
    main = torch.cuda.current_stream()
    own = [torch.cuda.Stream() for _ in range(n_streams)] or [main]
    theirs = torch.cuda.Stream()
    torch.cuda.synchronize()
    extra = None
    if foreign:
        with torch.cuda.stream(theirs):
            extra = sum((p.float() * 0.25).sum() for p in params)
    outs = []
    for i, x in enumerate(xs):
        with torch.cuda.stream(own[i % len(own)]):
            outs.append(_Slow.apply(layer(x.requires_grad_())[0]))
    torch.cuda.synchronize()
    outs[0].backward(dy)
    outs[1].backward(dy)
    torch.autograd.backward([outs[2], outs[3]] + ([extra] if foreign else []), [dy, dy] + ([None] if foreign else []))
    got = [p.grad.clone() for p in params]      # on the calling stream, which has waited for nothing by itself
    torch.cuda.synchronize()
    for p, g, *r in zip(params, got, *refs):
        assert torch.equal(p.grad, g)
        assert_close(g, sum(t.double() for t in r) + (0.25 if foreign else 0.0), torch.float16, "sum over four", 0.3)
    # (in the third backward the later forward comes first)
    assert added == ([0] * 4 if foreign else {0: [0, 1, 1, 1], 1: [0, 1, 1, 1], 2: [0, 0, 0, 1], 3: [0, 0, 1, 0]}[n_streams])


@pytest.mark.gpu
def test_slice_loop_adds_in_the_kernels(monkeypatch):
    """Slices of one sequence: the last one leaves .grad, every other one adds to it, layer by layer."""
    import terapipe_amd as ta
    from terapipe_amd import _layer_core as core
    from terapipe_amd import _lib
    from tests.util import reference_style_loop
    added = []
    native = core.layer_bwd_native

    def noted(image, device):
        added.append(_lib.LayerBwdDesc.from_buffer(image).wg_accumulate)
        native(image, device)

    monkeypatch.setattr(core, "layer_bwd_native", noted)
    layers = ta.TransformerLayers(2, 128, 512, 2, dtype=torch.float16)
    x = torch.randn(24, 1, 128, device="cuda").half()
    reference_style_loop(layers, x, torch.randn_like(x), [1], [8, 8, 8])
    assert added == [0, 0, 1, 1, 1, 1]
