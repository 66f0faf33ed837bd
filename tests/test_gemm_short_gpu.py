"""A group of weight gradients over few rows (tiles of 128 x 128, two workgroups per CU) at its edges: fewer k-tiles than stages, rows
and columns that end inside a tile, results stored and added, members of very different size; against fp64, and nothing written
beside the matrices."""
import ctypes

import pytest
import torch

from tests.util import assert_close

DEV = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("add", [False, True], ids=["store", "add"])
@pytest.mark.parametrize("K", [64, 128, 192, 512, 768])
def test_short_group(K, add, dtype):
    from terapipe_amd import _lib as L
    from terapipe_amd import ops
    g = torch.Generator(device=DEV).manual_seed(K)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    items, whole = [], []
    shapes = ((4800, 1600), (1000, 2056), (8, 8), (3016, 4504)) if K < 512 else ((4808, 1608), (1608, 1608), (6408, 1600), (1600, 6408))
    for M, N in shapes:
        buf = rnd(M + 2, N + 16).to(dtype)
        whole.append((buf, buf.clone()))
        items.append((L.TP_GEMM_TN, (rnd(K, M) * 0.1).to(dtype), rnd(K, N).to(dtype), M, N, K, buf[1:M + 1, 8:N + 8],
                      L.TP_EPI_ACCUMULATE if add else L.TP_EPI_STORE))
    sinks = [[] for _ in items]
    ops.gemm_grouped(items, desc_sinks=sinks)
    descs = (L.GemmDesc * len(items))(*(s[0] for s in sinks))
    rows, columns = ctypes.c_int(), ctypes.c_int()
    assert L.load().tp_gemm_group_tile(descs, len(items), ctypes.byref(rows), ctypes.byref(columns)) == 0
    assert (rows.value, columns.value) == (128, 128)
    for (op, a, b, M, N, K, c, _), (buf, old) in zip(items, whole):
        want = a.double().t() @ b.double() + (old[1:M + 1, 8:N + 8].double() if add else 0)
        assert_close(c, want, dtype, "%dx%d" % (M, N))
        buf[1:M + 1, 8:N + 8] = old[1:M + 1, 8:N + 8]
        assert torch.equal(buf, old)
