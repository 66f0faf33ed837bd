"""Products of a handful of rows (gemm_skinny_kernel): tiles of 8 and of 16 weight rows, k that ends inside a turn or a wave's
share, weights larger and smaller than the chip, and layer calls whose products take the LayerNorm before them too."""
import pytest
import torch

import oracle
from tests.util import assert_close, load_params_into, make_params, reference_style_loop

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("M,N,K", [
    (1, 8, 8), (8, 24, 72), (5, 1000, 40), (3, 2048, 2048), (8, 2048, 4104), (7, 2056, 1032), (1, 520, 8200), (8, 1024, 16384),
    (4, 6144, 2056), (2, 8200, 520), (6, 20488, 968), (8, 4096, 8200), (1, 7680, 2560), (9, 2048, 2056), (16, 1000, 1032), (17, 264, 2048),
    (32, 4104, 264)], ids=str)
@pytest.mark.parametrize("no_backward", [False, True])
def test_products(M, N, K, no_backward, dtype):
    from terapipe_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    A, B, bias, res = rnd(M, K), rnd(N, K) * K ** -0.5, rnd(N), rnd(M, N)
    want = A.double() @ B.double().t() + bias.double()
    C = torch.full((M + 1, N), 7.0, device=DEV, dtype=dtype)
    ops.gemm(ops.TP_GEMM_NT, A, B, M, N, K, C=C[:M], epilogue=ops.TP_EPI_BIAS, bias=bias, no_backward=no_backward)
    assert_close(C[:M], want, dtype, "bias")
    assert (C[M] == 7).all()
    ops.gemm(ops.TP_GEMM_NT, A, B, M, N, K, C=C[:M], epilogue=ops.TP_EPI_BIAS_RESIDUAL, bias=bias, residual=res,
             no_backward=no_backward)
    assert_close(C[:M], want + res.double(), dtype, "bias and residual")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("E,F,heads,batch,slices", [
    (128, 512, 2, 1, [1, 3, 8, 1]), (768, 3072, 12, 2, [1, 4, 2]), (640, 2560, 8, 3, [2, 1]), (2560, 16384, 32, 8, [1, 1]),
    (2304, 576, 18, 1, [2, 5, 9])], ids=str)
def test_layers_of_few_rows(E, F, heads, batch, slices, dtype):
    """One to nine rows a slice, forward and backward: what a fused launch leaves for the backward (the normalised rows, their
    statistics) enters every gradient."""
    import terapipe_amd as ta
    L = sum(slices)
    ps = make_params(2, E, F, dtype, seed=E)
    g = torch.Generator().manual_seed(L)
    x, dy = (torch.randn(L, batch, E, generator=g).to(dtype) for _ in range(2))
    layers = ta.TransformerLayers(2, E, F, heads, mixed_precision=True, dtype=dtype, device=DEV, activation="gelu")
    load_params_into(layers, ps, dtype)
    y, dx, _, _ = reference_style_loop(layers, x.to(DEV), dy.to(DEV), [batch], slices)
    leaf = [{k: v.clone().requires_grad_(True) for k, v in p.items()} for p in ps]
    yo, dxo, _ = oracle.terapipe_forward_backward(leaf, x.float(), dy.float(), heads, [batch], slices, activation="gelu")
    assert_close(y, yo, dtype, "y")
    assert_close(dx, dxo, dtype, "dx")
    for layer, p in zip(layers.layers, leaf):
        for name, t in layer.param_dict().items():
            assert_close(t.grad, p[name].grad, dtype, name)
    # the same slices without gradients
    with torch.no_grad():
        cache, done, out = layers.create_cache(batch, L), 0, []
        for n in slices:
            o, cache = layers(x[done:done + n].to(DEV), cache, done)
            out.append(o)
            done += n
    assert_close(torch.cat(out), yo, dtype, "y, forward only")
