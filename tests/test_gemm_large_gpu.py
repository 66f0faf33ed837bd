"""The 256 x 256 tile of eight waves and the pipelined tiles on a k that is no whole number of 64-wide k-tiles, against the
fp64 product."""
import pytest
import torch

from tests.util import assert_close

DEV = "cuda"
WIDE = 44


def _run(op, M, N, K, dtype, cfg=None, ksplit=None):
    from terapipe_amd import _lib as L
    from terapipe_amd import ops
    code = {"NT": L.TP_GEMM_NT, "NN": L.TP_GEMM_NN, "TN": L.TP_GEMM_TN}[op]
    g = torch.Generator(device=DEV).manual_seed(M + 3 * N + 7 * K)
    A = torch.randn((K, M) if op == "TN" else (M, K), generator=g, device=DEV).to(dtype)
    B = (torch.randn((N, K) if op == "NT" else (K, N), generator=g, device=DEV) * 0.1).to(dtype)
    C = torch.full((M, N), float("nan"), dtype=dtype, device=DEV)
    ops.gemm(code, A, B, M, N, K, C=C, tile_cfg=cfg, ksplit=ksplit)
    ref = (A.double().t() if op == "TN" else A.double()) @ (B.double().t() if op == "NT" else B.double())
    assert_close(C, ref, dtype, "%s %dx%dx%d" % (op, M, N, K))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("op", ["NT", "NN"])
@pytest.mark.parametrize("M,N,K,ksplit", [
    (256, 256, 64, 1), (256, 256, 128, 1), (256, 256, 192, 1),      # one, two, three k-tiles
    (1, 8, 64, 1), (257, 264, 320, 1), (511, 1000, 448, 1),         # edges inside a tile
    (300, 520, 1024, 3),                                            # k splits of unequal length
], ids=str)
def test_wide_tile(op, M, N, K, ksplit, dtype):
    _run(op, M, N, K, dtype, WIDE, ksplit)


@pytest.mark.gpu
@pytest.mark.parametrize("op,M,N,K", [
    ("NT", 4096, 4096, 1032), ("NN", 4096, 4096, 1032),             # the wide tile, 8 positions over
    ("NT", 1024, 5120, 200), ("NN", 1032, 5000, 184),               # the pipelined tiles
    ("NT", 520, 4096, 56), ("NN", 520, 4096, 56),                   # less than one k-tile
    ("TN", 4096, 4096, 1), ("TN", 4104, 4096, 257), ("TN", 1600, 1608, 333), ("TN", 2048, 6144, 95),
    ("NT", 200, 4096, 2088), ("NN", 200, 12288, 4104),              # slices of up to 512 rows
], ids=str)
def test_ragged_k(op, M, N, K):
    _run(op, M, N, K, torch.float16)


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["NT", "NN", "TN"])
def test_ragged_k_split(op):
    """A last split that is shorter than a k-tile."""
    _run(op, 600, 800, 1024 + 40, torch.bfloat16, ksplit=None)
    _run(op, 2048, 1024, 8192 + 24, torch.float16)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (1, 2048, 2048), (5, 24, 264), (16, 1000, 2056), (17, 4096, 1024), (31, 520, 5128),
                                   (4, 2048, 8192), (3, 15360, 1032), (32, 16, 40)], ids=str)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
def test_few_rows(M, N, K, dtype):
    """The kernel for up to 32 rows: one, two and four weight tiles per workgroup, a short last one, k tails, k splits."""
    _run("NT", M, N, K, dtype)
    _run("NT", M, N, K, dtype, None, 3 if K >= 192 else 1)
