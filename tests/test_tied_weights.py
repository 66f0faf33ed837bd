"""How an LM head's weight gradient reaches the embedding that shares the weight (CPU: the kernels are replaced by torch)."""
import pytest
import torch

V, E, M = 50, 8, 6
IDS = torch.tensor([3, 7, 3, 0, 49, 11])
DLOGITS = torch.linspace(-1, 1, M * V).view(M, V)


@pytest.fixture
def calls(monkeypatch):
    """Plain torch in place of the library; the calls made since the last look (`rows`: embedding rows added to something,
    `zeros`: into a gradient of their own)."""
    from terapipe_amd import ops
    from terapipe_amd._lib import TP_EPI_ACCUMULATE, TP_GEMM_NN, TP_GEMM_NT
    made = []

    def gemm(op, A, B, m, n, k, C, epilogue=0, ragged=False):
        if op not in (TP_GEMM_NT, TP_GEMM_NN):
            made.append("add" if epilogue == TP_EPI_ACCUMULATE else "dw")
        a, b = (A[:, :k], B.t()) if op == TP_GEMM_NT else (A[:, :k], B) if op == TP_GEMM_NN else (A[:, :m].t(), B)
        C[:, :n] = a @ b + (C[:, :n] if epilogue == TP_EPI_ACCUMULATE else 0)

    def rows(ids, dout, dw):
        made.append("rows" if dw.any() else "zeros")
        return dw.index_add_(0, ids, dout)

    def stream():
        return stream.now

    stream.now = 0
    for name, f in (("gemm", gemm), ("embedding_fwd", lambda ids, w: w[ids].clone()), ("embedding_bwd_rows_", rows),
                    ("zero_", lambda t: t.zero_()), ("embedding_bwd", lambda ids, d, acc: acc.index_add_(0, ids, d.float())),
                    ("accum_cast", lambda dst, src, add: dst.copy_(src + dst if add else src)), ("_stream", stream)):
        monkeypatch.setattr(ops, name, f)

    def look():
        out = list(made)
        made.clear()
        return out

    look.stream = stream
    return look


def _embedding():
    import terapipe_amd as ta
    torch.manual_seed(0)
    return ta.VocabParallelEmbedding(V, E, dtype=torch.float32)


def _head(h, w):
    import terapipe_amd as ta
    return (ta.lm_head_logits(h, w)[:, :V] * DLOGITS).sum()


def _hidden(seed=1):
    return torch.randn(M, E, generator=torch.Generator().manual_seed(seed)).requires_grad_()


def _expected(w, lookups=(), heads=()):
    """Gradient of sum(k * lookup) over `lookups` and of a head on every input of `heads`."""
    w = w.detach().clone().requires_grad_()
    total = sum((w[IDS] * k).sum() for k in lookups) + sum(((h.detach() @ w.t()) * DLOGITS).sum() for h in heads)
    return torch.autograd.grad(total, w)[0]


def _same(got, ref):
    assert torch.allclose(got, ref, rtol=1e-5, atol=1e-5), (got - ref).abs().max()


def test_model(calls):
    """Tokens through the embedding to the head: one dense gradient; accumulated over two passes; seen whole by a hook and by
    torch.autograd.grad."""
    emb = _embedding()
    loss = lambda: _head(emb(IDS) * 3, emb.weight)
    w = emb.weight.detach().clone().requires_grad_()
    ref, = torch.autograd.grad(((w[IDS] * 3 @ w.t()) * DLOGITS).sum(), w)
    for times in (1, 2):
        loss().backward()
        _same(emb.weight.grad, times * ref)
        assert calls() == ["dw", "rows"]
    _same(torch.autograd.grad(loss(), emb.weight)[0], ref)
    assert calls() == ["dw", "rows"]
    seen = []
    handle = emb.weight.register_hook(lambda g: seen.append(g.clone()))
    loss().backward()
    handle.remove()
    _same(seen[0], ref)
    assert len(seen) == 1 and calls() == ["dw", "rows"]
    y = loss()
    y.backward(retain_graph=True)
    y.backward()
    _same(emb.weight.grad, 5 * ref)
    assert calls() == ["dw", "rows"] * 2


def test_roots_of_their_own(calls):
    """Nothing but the weight ties them together: whichever runs first."""
    emb, h = _embedding(), _hidden()
    for order in ("embedding first", "head first"):     # the later forward runs its backward first
        emb.weight.grad = None
        if order == "embedding first":
            y, e = _head(h, emb.weight), emb(IDS)
        else:
            e, y = emb(IDS), _head(h, emb.weight)
        torch.autograd.backward([y, e], [None, torch.full_like(e, 2.0)])
        _same(emb.weight.grad, _expected(emb.weight, [2.0], [h]))
        assert calls() == (["zeros", "dw"] if order == "embedding first" else ["dw", "rows"])


def test_an_embedding_that_does_not_run(calls):
    """Its output is not part of the pass, or nothing below the head is asked for; then of a later pass."""
    emb, h = _embedding(), _hidden()
    e, y = emb(IDS), _head(h, emb.weight)
    y.backward(retain_graph=True)
    _same(emb.weight.grad, _expected(emb.weight, [], [h]))
    torch.autograd.grad(y, h, retain_graph=True)
    torch.autograd.grad(y + e.sum(), [h, e], retain_graph=True)
    torch.autograd.backward([y, e.sum()], inputs=[h, emb.weight])
    _same(emb.weight.grad, _expected(emb.weight, [1.0], [h, h]))
    del e
    emb.weight.grad = None
    _head(h, emb.weight).backward()
    _same(emb.weight.grad, _expected(emb.weight, [], [h]))


def test_several_heads_and_lookups(calls):
    emb, hs = _embedding(), [_hidden(i) for i in range(3)]
    es = [emb(IDS), emb(IDS)]
    ys = [_head(h, emb.weight) for h in hs]
    torch.autograd.backward(ys + es, [None] * 3 + [torch.full_like(es[0], k) for k in (2.0, 5.0)])
    _same(emb.weight.grad, _expected(emb.weight, [2.0, 5.0], hs))
    assert sorted(calls()) == ["add", "add", "dw", "rows", "zeros"]


def test_another_stream_and_a_graph_of_the_backward(calls):
    emb, h = _embedding(), _hidden()
    e = emb(IDS)
    y = _head(h, emb.weight)
    calls.stream.now = 5
    torch.autograd.backward([y, e], [None, torch.ones_like(e)], retain_graph=True)
    _same(emb.weight.grad, _expected(emb.weight, [1.0], [h]))
    assert sorted(calls()) == ["dw", "zeros"]
    calls.stream.now = 0
    got, = torch.autograd.grad([y, e], emb.weight, [torch.ones_like(y), torch.ones_like(e)], create_graph=True)
    _same(got, _expected(emb.weight, [1.0], [h]))
    assert sorted(calls()) == ["dw", "zeros"]


def test_a_pass_that_broke_off(calls):
    """What was handed over in it is forgotten."""
    emb, h = _embedding(), _hidden()

    class Breaks(torch.autograd.Function):
        broken = True

        @staticmethod
        def forward(ctx, x):
            return x.clone()

        @staticmethod
        def backward(ctx, g):
            if Breaks.broken:
                raise ValueError("broken")
            return g

    e = emb(IDS)
    total = Breaks.apply(e).sum() + _head(h, emb.weight)
    with pytest.raises(ValueError, match="broken"):
        total.backward(retain_graph=True)
    Breaks.broken = False
    emb.weight.grad = None
    total.backward()
    _same(emb.weight.grad, _expected(emb.weight, [1.0], [h]))


def test_other_weights_and_a_weight_that_is_no_leaf(calls):
    emb, other, h = _embedding(), _embedding(), _hidden()
    e, y = emb(IDS), _head(h, other.weight)
    (e.sum() + y).backward()
    _same(emb.weight.grad, _expected(emb.weight, [1.0]))
    _same(other.weight.grad, _expected(emb.weight, [], [h]))
    assert sorted(calls()) == ["dw", "zeros"]
    base = emb.weight.detach().clone().requires_grad_()
    both = base * 1.0
    del emb.weight
    emb.weight = both
    (emb(IDS).sum() + _head(h, both)).backward()
    _same(base.grad, _expected(both, [1.0], [h]))
    assert calls() == ["dw", "rows"]


@pytest.mark.parametrize("tied", [False, True])
def test_rows_that_do_not_fit(calls, tied, monkeypatch):
    """The fp32 path of lookups that are too long for the row kernel adds to what it is handed as well."""
    from terapipe_amd import ops
    monkeypatch.setattr(ops, "embedding_rows_fit", lambda ids, dout: False)
    emb, h = _embedding(), _hidden()
    e = emb(IDS)
    (e.sum() + (_head(h, emb.weight) if tied else 0)).backward()
    _same(emb.weight.grad, _expected(emb.weight, [1.0], [h] if tied else []))


def test_nothing_is_kept_alive(calls):
    """A weight whose AccumulateGrad node lives on does not collect the lookups of past steps."""
    from terapipe_amd import _autograd
    emb = _embedding()
    node = torch.autograd.graph.get_gradient_edge(emb.weight).node
    for _ in range(5):
        emb(IDS).sum().backward()
    assert len(node.metadata[_autograd._LOOKUPS]) == 1


def test_a_lookup_nobody_noted(calls):
    """The autograd function by itself, without the module."""
    from terapipe_amd import vocab
    emb, h = _embedding(), _hidden()
    (vocab._EmbeddingFunction.apply(IDS, emb.weight).sum() + _head(h, emb.weight)).backward()
    _same(emb.weight.grad, _expected(emb.weight, [1.0], [h]))
    assert sorted(calls()) == ["dw", "zeros"]
