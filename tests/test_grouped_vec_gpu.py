"""Weight gradients and vector-parameter gradients of the same rows in one call: as blocks of one launch behind its tiles of 256 x 256,
or in two launches where the products run on other tiles or one by one."""
import ctypes

import pytest
import torch

from tests.util import assert_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype,E,F,M,tile", [
    (torch.float16, 1024, 4096, 1024, 256), (torch.bfloat16, 904, 3608, 1088, 256), (torch.float16, 1016, 4056, 832, 256),     # one launch
    (torch.float16, 2048, 8192, 832, 256), (torch.bfloat16, 520, 2056, 1088, 128), (torch.float16, 768, 3072, 128, 128),
    (torch.float16, 264, 520, 1000, 0), (torch.float32, 256, 1024, 320, 0)], ids=str)
def test_as_two_calls(dtype, E, F, M, tile):
    from terapipe_amd import _lib as L
    from terapipe_amd import ops
    g = torch.Generator(device=DEV).manual_seed(E + M)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    dqkv, dh, dz1, dout, xn, o, hn, a = (rnd(M, w) for w in (3 * E, E, F, E, E, E, E, F))
    dxn, dhn, x, h = (rnd(M, E) for _ in range(4))
    mean, rstd = torch.randn(2, M, generator=g, device=DEV)
    rstd = rstd.abs()

    def both(together):
        out = [torch.full(s, 7.0, device=DEV, dtype=dtype) for s in ((3 * E, E), (E, E), (F, E), (E, F))]
        items = [(L.TP_GEMM_TN, dy, xi, dy.shape[1], xi.shape[1], M, c, L.TP_EPI_STORE)
                 for dy, xi, c in zip((dqkv, dh, dz1, dout), (xn, o, hn, a), out)]
        acc = [torch.ones(n, device=DEV) for n in (3 * E, E, F, E, E, E, E, E)]
        vecs = [(dqkv, acc[0]), (dh, acc[1]), (dz1, acc[2]), (dout, acc[3]), (dxn, x, mean, rstd, acc[4], acc[5]),
                (dhn, h, mean, rstd, acc[6], acc[7])]
        sinks = [[] for _ in items]
        if together:
            ops.gemm_grouped(items, sinks, vecs)
        else:
            ops.gemm_grouped(items, sinks)
            ops.vec_param_grads(vecs)
        descs = (L.GemmDesc * 4)(*[s[0] for s in sinks])
        rows = ctypes.c_int()
        L.load().tp_gemm_group_tile(descs, 4, ctypes.byref(rows), None)
        return out, acc, rows.value

    want, _, rows = both(False)
    got, acc, _ = both(True)
    assert rows == tile
    assert all(torch.equal(p, q) for p, q in zip(got, want))
    xhat = [(t.double() - mean.double()[:, None]) * rstd.double()[:, None] for t in (x, h)]
    sums = [t.double().sum(0) for t in (dqkv, dh, dz1, dout)] + [
        (dxn.double() * xhat[0]).sum(0), dxn.double().sum(0), (dhn.double() * xhat[1]).sum(0), dhn.double().sum(0)]
    for i, (p, q) in enumerate(zip(acc, sums)):
        assert_close(p, q + 1, torch.float32, "sum %d" % i)
