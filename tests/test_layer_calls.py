"""Whole layers per library call: descriptor layouts (CPU), the forward-only stack and the two ways parameter gradients reach
.grad on the layer-level surface (GPU)."""
import ctypes
import os
import subprocess

import pytest
import torch

from tests.util import assert_close

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_descriptor_layouts(tmp_path):
    from terapipe_amd import _layer_core as core
    from terapipe_amd import _lib
    src = tmp_path / "t.c"
    src.write_text(r'''
#include <stdio.h>
#include <stddef.h>
#include "terapipe_hip.h"
int main(void) {
  printf("%zu %zu %zu %zu %zu %zu\n", sizeof(tp_layer_desc), offsetof(tp_layer_desc, x), offsetof(tp_layer_desc, out),
         sizeof(tp_layer_bwd_desc), offsetof(tp_layer_bwd_desc, wg_rows), offsetof(tp_layer_bwd_desc, small_out));
  return 0;
}''')
    exe = str(tmp_path / "t")
    subprocess.check_call(["gcc", "-I", os.path.join(ROOT, "include"), str(src), "-o", exe])
    got = [int(v) for v in subprocess.check_output([exe]).split()]
    L, B = _lib.LayerDesc, _lib.LayerBwdDesc
    assert got == [ctypes.sizeof(L), L.x.offset, L.out.offset, ctypes.sizeof(B), B.wg_rows.offset, B.small_out.offset]
    assert core._FWD_PACK.size == ctypes.sizeof(L) and core._FWD_PACK.size + core._BWD_PACK.size == ctypes.sizeof(B)


def test_bad_descriptors_are_refused():
    from terapipe_amd import _lib
    lib = _lib.load()
    d = _lib.LayerDesc()
    assert lib.tp_layers_fwd(ctypes.addressof(d), 1, None, 0, None) == 1 and b"bad sizes" in lib.tp_last_error()
    d.T, d.batch, d.heads, d.hidden, d.ffn, d.cache_rows = 4, 1, 1, 64, 256, 4
    assert lib.tp_layers_fwd(ctypes.addressof(d), 1, None, 0, None) == 1 and b"parameter 0" in lib.tp_last_error()
    assert lib.tp_layer_bwd(None, None, 0, None) == 1


def _stack(nl, E, H, dtype, activation="gelu"):
    import terapipe_amd as ta
    torch.manual_seed(3)
    layers = ta.TransformerLayers(nl, E, 4 * E, H, dtype=dtype, device="cuda", activation=activation)
    with torch.no_grad():
        for p in layers.parameters():
            p.add_(torch.randn_like(p) * 0.02)
    return layers


@pytest.mark.gpu
@pytest.mark.parametrize("nl,E,H,B,T,P,dtype", [
    (1, 128, 2, 2, 5, 3, torch.float16), (2, 128, 1, 1, 1, 40, torch.bfloat16), (5, 256, 2, 3, 33, 0, torch.float16),
    (3, 160, 2, 1, 7, 9, torch.float16), (3, 128, 2, 2, 9, 4, torch.float32)], ids=str)
def test_forward_only_stack_gives_the_layers_bits(nl, E, H, B, T, P, dtype):
    layers = _stack(nl, E, H, dtype)
    x = torch.randn(T, B, E, device="cuda").to(dtype)
    caches = [torch.randn_like(c) for c in layers.create_cache(B, P + T + 2)]
    kept = [c.clone() for c in caches]
    y, out = layers(x, [c.requires_grad_() for c in kept], P)
    with torch.no_grad():
        y0, out0 = layers(x, caches, P)
    assert not y0.requires_grad and [c.data_ptr() for c in out0] == [c.data_ptr() for c in caches]
    # between two layers the LayerNorm may add the k-split sums of fc2 itself: the same sum, rounded once
    assert_close(y0, y, dtype, "y", 1.0 if dtype == torch.float32 else 0.1)
    for a, b in zip(out0, out):
        assert_close(a, b, dtype, "cache", 1.0 if dtype == torch.float32 else 0.1)
    layer = layers.layers[0]
    ref, none = layer(x.detach().requires_grad_())
    with torch.no_grad():
        got, none0 = layer(x)
    assert none is None and none0 is None and torch.equal(got, ref)


@pytest.mark.gpu
def test_parameter_gradients_with_and_without_the_kernels_adding_them():
    """A second backward adds to .grad inside the kernels; autograd.grad, backward(inputs=...), and hooks see gradients as
    tensors and leave .grad to autograd."""
    layers = _stack(1, 128, 2, torch.float16)
    layer, params = layers.layers[0], list(layers.parameters())
    x = torch.randn(16, 2, 128, device="cuda").half()
    dy = torch.randn_like(x)
    run = lambda: layer(x.clone().requires_grad_())[0]
    run().backward(dy)
    once = [p.grad.clone() for p in params]
    where = [p.grad.data_ptr() for p in params]
    run().backward(dy)
    for p, g, at in zip(params, once, where):
        assert p.grad.data_ptr() == at
        assert_close(p.grad, 2 * g.float(), torch.float16, "two backward passes", 0.1)
    twice = [p.grad.clone() for p in params]
    for g, h in zip(torch.autograd.grad(run(), params, dy), once):
        assert_close(g, h, torch.float16, "autograd.grad", 0.1)
    xi = x.clone().requires_grad_()
    torch.autograd.backward([layer(xi)[0]], [dy], inputs=[xi])
    assert xi.grad is not None and all(torch.equal(p.grad, g) for p, g in zip(params, twice))
    seen = []
    handle = params[2].register_hook(lambda g: seen.append(g.clone()))
    run().backward(dy)
    handle.remove()
    assert len(seen) == 1 and seen[0] is not None
    assert_close(seen[0], once[2], torch.float16, "hook", 0.1)
    assert_close(params[2].grad, 3 * once[2].float(), torch.float16, "three backward passes", 0.1)
