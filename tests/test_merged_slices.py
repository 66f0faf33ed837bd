"""The pieces a runner's step runs in: the rule on the CPU, and merged steps against the CPU oracle."""
import pytest
import torch

import oracle
from tests.util import assert_close, load_params_into, make_params


def test_rule():
    from terapipe_amd.terapipe import merges
    assert merges(None) and not any(merges(n) for n in (1, 2, 3))


def test_who_merges():
    import terapipe_amd as ta
    layers = ta.TransformerLayers(1, 64, 128, 1, dtype=torch.float16, device="cpu")
    make = lambda bs=(2,), **kw: ta.TeraPipe(layers, 2, 64, list(bs), [32, 32], **kw).merge_slices
    assert make() and make(launch_replay=False) and make(slice_streams=1, merge_slices=True)
    assert not any(make(**kw) for kw in (dict(slice_streams=3), dict(slice_streams=1), dict(use_hip_graph=True),
                                         dict(suffix_dkdv=False), dict(fp32_grad_cache=False), dict(bs=(1, 1)), dict(merge_slices=False)))


@pytest.mark.gpu
def test_one_stream_runs_the_slices():
    """Slices that somebody asks for run one by one also where they are long and the weights small (eight of 256 rows of
    hidden 2048)."""
    import terapipe_amd as ta
    layers = ta.TransformerLayers(1, 2048, 2048, 16, dtype=torch.float16)
    x = torch.randn(2048, 1, 2048, device="cuda").half()
    for kw, pieces in ((dict(slice_streams=1), [256] * 8), (dict(merge_slices=False), [256] * 8), (dict(), [2048])):
        runner = ta.TeraPipe(layers, 1, 2048, [1], [256] * 8, **kw)
        runner(x).sum().backward()
        assert runner._sbufs.pieces == pieces and len(runner._sbufs.lanes) == (2 if kw.get("merge_slices") is False else 0)


@pytest.mark.gpu
@pytest.mark.parametrize("E,H,B,slices,dtype,pieces", [
    (128, 2, 3, [7, 1, 30, 27], torch.float16, [65]),             # odd length
    (128, 1, 32, [33, 31, 5], torch.bfloat16, [69]),              # more than 2048 rows
    (160, 2, 16, [100, 31], torch.float16, [131]),                # head dimension 80
    (128, 2, 3, [7, 1, 30, 27], torch.float32, [65]),             # gradient caches
], ids=str)
def test_merged_step_against_the_oracle(E, H, B, slices, dtype, pieces):
    """Three steps (eager, recorded, re-issued) of the default runner, GeLU so that no sign decision is involved."""
    import terapipe_amd as ta
    L, nl = sum(slices), 2
    ps = make_params(nl, E, 4 * E, dtype, seed=5)
    layers = ta.TransformerLayers(nl, E, 4 * E, H, dtype=dtype, device="cuda", activation="gelu")
    load_params_into(layers, ps, dtype)
    runner = ta.TeraPipe(layers, B, L, [B], slices)
    g = torch.Generator().manual_seed(9)
    x, dy = torch.randn(L, B, E, generator=g).to(dtype), torch.randn(L, B, E, generator=g).to(dtype)
    leaf = [{k: v.clone().requires_grad_(True) for k, v in p.items()} for p in ps]
    yo, dxo, _ = oracle.terapipe_forward_backward(leaf, x.float(), dy.float(), H, [B], slices, activation="gelu")
    for step in range(3):
        for p in layers.parameters():
            p.grad = None
        xd = x.cuda().requires_grad_(True)
        y = runner(xd)
        y.backward(dy.cuda())
        assert runner._sbufs.pieces == pieces
        assert_close(y, yo, dtype, "step %d: y" % step)
        assert_close(xd.grad, dxo, dtype, "step %d: dx" % step)
        for l, layer in enumerate(layers.layers):
            for name, p in layer.param_dict().items():
                assert_close(p.grad, leaf[l][name].grad, dtype, "step %d: layer %d %s" % (step, l, name))
