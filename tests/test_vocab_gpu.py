"""The kernels of the two ends of the stack at their edges: gradient rows of the embedding, loss and gradient of the
cross-entropy, products over a vocabulary that is no multiple of 8, and where their gradients end up."""
import pytest
import torch
import torch.nn.functional as F

from tests.util import assert_close

DEV = "cuda"
DTYPES = pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=str)
pytestmark = pytest.mark.gpu


@DTYPES
@pytest.mark.parametrize("M,E,V", [(1, 8, 1), (511, 264, 3), (513, 2056, 700), (1100, 16, 2000), (8192, 64, 5)], ids=str)
def test_embedding_rows(dtype, M, E, V):
    from terapipe_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M)
    ids = torch.randint(-1, V + 1, (M,), generator=g, device=DEV)       # ids outside the vocabulary add nothing
    dout = (torch.randn(M, E, generator=g, device=DEV) / 16).to(dtype)
    dw = torch.randn(V, E, generator=g, device=DEV).to(dtype)
    inside = (ids >= 0) & (ids < V)
    ref = dw.double().index_add(0, ids[inside], dout.double()[inside])
    ops.embedding_bwd_rows_(ids, dout, dw)
    assert_close(dw, ref, dtype, "rows")


@DTYPES
@pytest.mark.parametrize("M,V,ld,shift", [(1, 1, 8, 0), (3, 8192, 8192, 0), (5, 8191, 8200, 0), (2, 40001, 40064, 0),
                                          (7, 777, 779, 0), (4, 1000, 1008, 1)], ids=str)
def test_loss_and_gradient(dtype, M, V, ld, shift):
    """Whole and ragged chunks; rows of odd length and rows that are not aligned take the scalar kernels."""
    from terapipe_amd import ops
    g = torch.Generator(device=DEV).manual_seed(V)
    buf = (torch.randn(M * ld + shift, generator=g, device=DEV) * 3).to(dtype)
    z = buf[shift:].view(M, ld)
    target = torch.randint(0, V, (M,), generator=g, device=DEV)
    scale = torch.rand(M, generator=g, device=DEV)
    zr = z[:, :V].double().clone().requires_grad_(True)
    ref = F.cross_entropy(zr, target, reduction="none")
    (ref * scale.double()).sum().backward()
    loss, stats = ops.cross_entropy_loss(z, target, V)
    assert_close(loss, ref, torch.float32, "loss", 1.0 if dtype == torch.float32 else 10.0)
    ops.cross_entropy_grad_(z, target, stats, scale, V)
    assert_close(z[:, :V], zr.grad, dtype, "gradient")
    assert not z[:, V:].any()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("V", [1, 9, 257, 4097, 50257])
@pytest.mark.parametrize("M", [1, 40, 300])
def test_ragged_vocabulary(dtype, V, M):
    """N of NT, k of NN and M of TN, none a multiple of 8."""
    import terapipe_amd as ta
    E = 256
    g = torch.Generator(device=DEV).manual_seed(V + M)
    h = torch.randn(M, E, generator=g, device=DEV).to(dtype).requires_grad_(True)
    w = (torch.randn(V, E, generator=g, device=DEV) * 0.05).to(dtype).requires_grad_(True)
    logits = ta.lm_head_logits(h, w)
    assert not logits[:, V:].any()
    dl = torch.randn(logits.shape, generator=g, device=DEV).to(dtype)
    dl[:, V:] = 0
    logits.backward(dl)
    hd, wd = h.detach().double(), w.detach().double()
    assert_close(logits[:, :V], hd @ wd.t(), dtype, "logits")
    assert_close(h.grad, dl[:, :V].double() @ wd, dtype, "dh")
    assert_close(w.grad, dl[:, :V].double().t() @ hd, dtype, "dw")


@DTYPES
@pytest.mark.parametrize("tied", [False, True])
def test_where_gradients_go(dtype, tied):
    """Into fresh and into existing gradients, of tied and of separate weights, with autograd's hooks and with
    torch.autograd.grad: all the same sums."""
    import terapipe_amd as ta
    V, E, M = 203, 64, 90
    g = torch.Generator().manual_seed(3)
    emb = ta.VocabParallelEmbedding(V, E, device=DEV, dtype=dtype)
    head = emb.weight if tied else torch.nn.Parameter(torch.randn(V, E, generator=g).mul(0.1).to(dtype).to(DEV))
    params = [emb.weight] if tied else [emb.weight, head]
    ids, target = (torch.randint(0, V, (M,), generator=g).to(DEV) for _ in range(2))

    def loss():
        return ta.vocab_parallel_cross_entropy(ta.lm_head_logits(emb(ids) * 4, head), target, vocab_size=V).sum()

    ws = [p.detach().double().requires_grad_(True) for p in params]
    F.cross_entropy(F.embedding(ids, ws[0]) * 4 @ ws[-1].t(), target, reduction="sum").backward()
    for got, w in zip(torch.autograd.grad(loss(), params), ws):
        assert_close(got, w.grad, dtype, "torch.autograd.grad")
    assert all(p.grad is None for p in params)
    for times in (1, 2):
        loss().backward()
        for p, w in zip(params, ws):
            assert_close(p.grad, times * w.grad, dtype, "backward %d" % times)
    seen = []
    handle = params[0].register_hook(lambda t: seen.append(t.detach().clone()))
    loss().backward()
    handle.remove()
    assert_close(sum(seen), ws[0].grad, dtype, "what a hook sees")
    assert_close(params[0].grad, 3 * ws[0].grad, dtype, "backward with a hook")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=str)
@pytest.mark.parametrize("V", [1, 9, 50])
def test_products_next_to_other_values(dtype, V):
    """N of NT, k of NN and M of TN inside a chunk: a plain product refuses them, and one that says it may use the rest of
    the chunk writes C's columns up to the next multiple of 8 and none beyond, and depends on nothing it reads there."""
    from terapipe_amd import _lib, ops
    from terapipe_amd._lib import TP_GEMM_NN, TP_GEMM_NT, TP_GEMM_TN
    M, E, up = 40, 64, (V + 7) // 8 * 8
    g = torch.Generator(device=DEV).manual_seed(V)
    h, w = (torch.randn(n, E, generator=g, device=DEV).to(dtype) for n in (M, V))
    wide = torch.full((M, up + 8), 7.0, dtype=dtype, device=DEV)
    dl = torch.randn(M, up + 8, generator=g, device=DEV).to(dtype)
    with pytest.raises(_lib.TeraPipeHipError, match="multiple of 8"):
        ops.gemm(TP_GEMM_NT, h, w, M, V, E, C=wide)
    for op, A, B, m, n, k in ((TP_GEMM_NN, dl, w, M, E, V), (TP_GEMM_TN, dl, h, V, E, M)):
        with pytest.raises(_lib.TeraPipeHipError, match="must be multiples"):
            ops.gemm(op, A, B, m, n, k, C=torch.empty(m, n, dtype=dtype, device=DEV))
    ops.gemm(TP_GEMM_NT, h, w, M, V, E, C=wide, ragged=True)
    assert_close(wide[:, :V], h.double() @ w.double().t(), dtype, "NT")
    assert (wide[:, up:] == 7).all()
    dh, dw = torch.empty(M, E, dtype=dtype, device=DEV), torch.full((V + 1, E), 7.0, dtype=dtype, device=DEV)
    ops.gemm(TP_GEMM_NN, dl, w, M, E, V, C=dh, ragged=True)
    ops.gemm(TP_GEMM_TN, dl, h, V, E, M, C=dw[:V], ragged=True)
    assert_close(dh, dl[:, :V].double() @ w.double(), dtype, "NN")
    assert_close(dw[:V], dl[:, :V].double().t() @ h.double(), dtype, "TN")
    assert (dw[V:] == 7).all()


@DTYPES
@pytest.mark.parametrize("V,ld", [(5, 7), (40, 40), (1000, 1003), (2050, 2056), (33000, 33000)], ids=str)
def test_loss_of_infinities_nan_and_masks(dtype, V, ld):
    """Rows with +-infinity, NaN (one, a thread's whole share, all) and masks of the type's lowest value: loss and gradient as
    the fp64 softmax has them, NaN where it has NaN.  (Vectors and scalars, one thread's share and several.)"""
    from terapipe_amd import ops
    g = torch.Generator(device=DEV).manual_seed(V)
    inf, nan, low = float("inf"), float("nan"), torch.finfo(dtype).min
    share = slice(min(V - 1, 8), min(V, 16))
    changes = [(slice(0, 0), 0.), (slice(1, 2), -inf), (slice(0, V - 1), -inf), (slice(0, V), -inf), (slice(2, 3), inf),
               (slice(0, 2), inf), (slice(V - 1, V), nan), (share, nan), (slice(0, V), nan), (slice(0, V - 1), low),
               (share, low), (slice(0, V), low)]
    M = len(changes)
    z = torch.randn(M, ld, generator=g, device=DEV).to(dtype)
    for m, (where, value) in enumerate(changes):
        z[m, where] = value
    target = torch.full((M,), V - 1, device=DEV)
    scale = torch.rand(M, generator=g, device=DEV) + 0.5
    zd = z[:, :V].double()
    top = zd.max(1, keepdim=True).values
    p = (zd - top).exp()
    # (the maximum and the target's logit first: beside 3.4e38 a logarithm is lost in fp64 as well)
    ref = (top[:, 0] - zd[:, V - 1]) + p.sum(1).log()
    grad = p / p.sum(1, keepdim=True)
    grad[:, V - 1] -= 1
    grad *= scale.double()[:, None]
    bad = torch.isnan(grad).any(1)
    assert bad.tolist() == [m in (3, 4, 5, 6, 7, 8) for m in range(M)]
    loss, stats = ops.cross_entropy_loss(z, target, V)
    ops.cross_entropy_grad_(z, target, stats, scale, V)
    assert torch.isnan(loss[bad]).all() and torch.isnan(z[bad][:, :V]).all()
    assert_close(loss[~bad], ref[~bad], torch.float32, "loss", 1.0 if dtype == torch.float32 else 10.0)
    assert_close(z[~bad][:, :V], grad[~bad], dtype, "gradient")
    assert not z[:, V:].any()
