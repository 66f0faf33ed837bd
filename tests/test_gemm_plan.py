"""The GEMM plan (tile configuration + k splits) that tp_gemm picks, asked through tp_gemm_plan: host code, so these
run without a GPU.  The measured table must give every shape of the four benchmark geometries exactly its entry, and
the rules for slice GEMMs outside the table must give plans that are valid and that follow the stated principles
(one round of workgroups when k is split, no split that leaves less than 1536 of k)."""
import ctypes
import os
import re

import pytest

from terapipe_amd import _lib

OPS = {"NT": _lib.TP_GEMM_NT, "NN": _lib.TP_GEMM_NN, "TN": _lib.TP_GEMM_TN}
# tile configuration -> (rows, columns, workgroups that fit a CU)
TILES = {0: (64, 64, 2), 2: (256, 256, 1), 6: (192, 160, 1), 7: (160, 160, 1), 3: (128, 256, 1), 5: (128, 128, 2), 8: (64, 64, 2), 11: (64, 256, 1),
         12: (64, 64, 2), 13: (128, 128, 1), 14: (192, 128, 1), 15: (256, 128, 1), 16: (128, 128, 1), 17: (256, 160, 1), 18: (256, 128, 1), 19: (256, 256, 1), 20: (256, 256, 1),
         31: (192, 128, 1), 33: (192, 256, 1), 41: (224, 128, 1), 42: (160, 128, 1), 43: (224, 160, 1)}


def plan(op, M, N, K, dtype=_lib.TP_F16):
    d = _lib.GemmDesc()
    d.op, d.dtype, d.epilogue, d.M, d.N, d.K = OPS[op], dtype, _lib.TP_EPI_STORE, M, N, K
    d.A = d.B = d.C = 4096          # never dereferenced: the plan is host arithmetic on the extents
    d.lda = M if op == "TN" else K
    d.ldb = K if op == "NT" else N
    d.ldc = N
    c, n = ctypes.c_int(), ctypes.c_int()
    rc = _lib.load().tp_gemm_plan(ctypes.byref(d), ctypes.byref(c), ctypes.byref(n))
    assert rc == 0, _lib.load().tp_last_error()
    assert n.value == _lib.load().tp_gemm_splits(ctypes.byref(d))
    return c.value, n.value


def _table():
    path = os.path.join(os.path.dirname(_lib.__file__), "csrc", "gemm_tuned.inc")
    out = []
    for line in open(path):
        m = re.match(r"\{TP_GEMM_(\w+), (\d+), (\d+), (\d+), (\d+), (\d+)\}", line)
        if m:
            out.append((m.group(1),) + tuple(int(v) for v in m.groups()[1:]))
    return out


def test_every_table_entry_is_the_plan_of_its_shape():
    entries = _table()
    assert len(entries) >= 90
    for op, M, N, K, cfg, ns in entries:
        assert plan(op, M, N, K) == (cfg, ns), (op, M, N, K)
        assert plan(op, M, N, K, _lib.TP_BF16) == (cfg, ns), (op, M, N, K)


def test_the_baseline_geometries_are_covered_by_exact_entries():
    """Every 16-bit GEMM of benchmark configs 2-5 (slice linears at each slice length, parameter gradients of a step)
    has its own entry, so that a revision of the rules cannot move a benchmark shape."""
    have = {e[:4] for e in _table()}
    geos = [(2048, 8192, [256], 2048), (5120, 20480, [512, 384, 320, 256, 224, 192, 160], 2048),
            (12288, 49152, [128], 2048), (6144, 24576, [64], 4096)]
    for E, F, rows, step in geos:
        for N, K in ((3 * E, E), (E, E), (F, E), (E, F)):
            for M in rows:
                assert ("NT", M, N, K) in have and ("NN", M, K, N) in have, (M, N, K)
            assert ("TN", N, K, step) in have, (N, K, step)


@pytest.mark.parametrize("E,F", [(1024, 4096), (3072, 12288), (4096, 16384), (7168, 28672), (8192, 32768), (10240, 40960)])
def test_rules_for_slice_gemms_outside_the_table(E, F):
    for M in (8, 40, 64, 96, 128, 160, 200, 256, 320, 384, 448, 512):
        for N, K in ((3 * E, E), (E, E), (F, E), (E, F)):
            for op, n, k in (("NT", N, K), ("NN", K, N)):
                cfg, ns = plan(op, M, n, k)
                assert cfg in TILES, (op, M, n, k, cfg)
                bm, bn, per_cu = TILES[cfg]
                tiles = -(-M // bm) * -(-n // bn)
                assert 1 <= ns <= 8
                if ns > 1:
                    assert k // ns >= 1536, "split too thin: %s" % ((op, M, n, k, cfg, ns),)
                    assert tiles * ns <= 256 * per_cu, "more than one round of workgroups: %s" % ((op, M, n, k, cfg, ns),)
                # a tile is never taller than twice the slice
                assert bm < 2 * max(M, 64), (op, M, n, k, cfg)


def test_rule_examples():
    """Shapes from the sweeps the rules were drawn from (measured best or within a few percent of it)."""
    assert plan("NT", 64, 16384, 4096) == (8, 1)           # 256 tiles of 64 x 64
    assert plan("NN", 64, 4096, 16384) == (8, 4)           # 64 tiles, k split to 256 workgroups
    assert plan("NT", 128, 4096, 4096) == (12, 1)          # small weight: 64 x 64 x 128 tiles, unsplit
    assert plan("NN", 128, 4096, 12288) == (16, 8)         # 32 tiles of 128 x 128 (the pipelined tile)
    assert plan("NT", 256, 32768, 8192) == (3, 1)          # 256 tiles of 128 x 256
    assert plan("NN", 256, 8192, 32768) == (3, 4)          # 64 of them on a long k
    assert plan("NT", 256, 12288, 4096) == (16, 1)         # 192 tiles of 128 x 128, k too short to split
    assert plan("NT", 320, 30720, 10240) == (33, 1)        # two row tiles of 192: the weight-streaming kernel
    assert plan("NT", 512, 20480, 4096) == (19, 1)         # two rows of 256 x 256 tiles
    assert plan("NN", 512, 4096, 16384) == (15, 4)         # 2 x 32 pipelined tiles of 256 x 128 on a long k
    assert plan("NT", 384, 16384, 4096) == (14, 1)         # two row tiles of 192 x 128
    assert plan("NT", 224, 16384, 8192) == (41, 2)         # one row of 224 x 128 tiles: nothing of a tile beyond the slice
    assert plan("NN", 448, 8192, 32768) == (41, 2)         # two of them
    assert plan("NT", 320, 16384, 8192) == (42, 1)         # two row tiles of 160 x 128
    assert plan("NT", 160, 32768, 8192) == (42, 1)         # one
    # fp32 keeps its own plan (64 x 64 register-staged tiles)
    assert plan("NT", 128, 4096, 4096, _lib.TP_F32)[0] == 0


def test_entries_between_their_row_counts():
    """Small weights take an entry near its own row count only; on larger ones fewer row tiles mean more k splits."""
    assert plan("NT", 256, 6144, 2048) == (8, 1) and plan("NT", 256, 8192, 2048) == (16, 1)
    for M in (128, 160, 192):
        assert plan("NT", M, 6144, 2048)[0] in (8, 12) and plan("NT", M, 8192, 2048)[0] in (8, 12), M      # the estimate
    assert plan("NN", 160, 5120, 5120) == (16, 3)
    for M in (80, 112, 128):
        assert plan("NN", M, 5120, 5120) == (16, 6), M
    assert plan("NN", 129, 5120, 5120) == (16, 3)           # the same row tiles as 160
    d = _lib.GemmDesc()
    d.op, d.dtype, d.epilogue, d.M, d.N, d.K, d.reserved = OPS["NN"], _lib.TP_F16, _lib.TP_EPI_STORE, 128, 5120, 5120, 1 << 24
    d.A = d.B = d.C = 4096
    d.lda = d.ldb = d.ldc = 5120
    assert _lib.load().tp_gemm_splits(ctypes.byref(d)) == 4         # beside other streams: its own entry, as it is


def test_the_estimate_keeps_narrow_tiles_where_two_fit_a_cu():
    """64 x 64 tiles up to two per CU, not a third as many of 128 x 128 (8.2 to 9.7 us against 11.0 to 11.8)."""
    for op, M, N, K in (("NT", 640, 2304, 768), ("NT", 768, 2304, 768), ("NT", 1500, 1024, 1024), ("NN", 1500, 1024, 1024),
                        ("NT", 520, 2304, 768), ("NN", 768, 768, 2304), ("NN", 384, 4096, 1024), ("NN", 512, 3072, 768)):
        assert plan(op, M, N, K)[0] in (8, 12), (op, M, N, K)


def _forced_plan(op, M, N, K, cfg, nsplit=0):
    d = _lib.GemmDesc()
    d.op, d.dtype, d.epilogue, d.M, d.N, d.K = OPS[op], _lib.TP_F16, _lib.TP_EPI_STORE, M, N, K
    d.A = d.B = d.C = 4096
    d.lda = M if op == "TN" else K
    d.ldb = K if op == "NT" else N
    d.ldc = N
    d.reserved = (cfg + 1) | (nsplit << 8)
    c, n = ctypes.c_int(), ctypes.c_int()
    assert _lib.load().tp_gemm_plan(ctypes.byref(d), ctypes.byref(c), ctypes.byref(n)) == 0
    return c.value, n.value


def test_forced_tiles_that_load_whole_k_tiles_fall_back_on_a_ragged_k():
    """A tile configuration forced through the descriptor's reserved field is replaced by the 128 x 128 register-
    free tile (5) when the kernel behind it cannot run the shape: the weight-streaming, pipelined and tall tiles
    load whole 64-wide k-tiles only, the weight-streaming tiles have no TN form."""
    for cfg in (21, 26, 33, 40, 14, 15, 16, 19, 2, 41, 42, 43):
        assert _forced_plan("NT", 128, 1024, 1024, cfg)[0] == cfg, cfg          # K % 64 == 0: taken as forced
        assert _forced_plan("NT", 128, 1024, 72, cfg)[0] == 5, cfg              # K = 72: would drop the k tail
        assert _forced_plan("NN", 128, 1024, 1096, cfg)[0] == 5, cfg
    for cfg in (21, 33, 41, 42, 43):
        assert _forced_plan("TN", 1024, 1024, 1024, cfg)[0] == 5, cfg
    assert _forced_plan("NN", 128, 1024, 1024, 24)[0] == 5                      # 80-wide tiles: NT only
    assert _forced_plan("NN", 224, 1024, 1024, 43)[0] == 5                      # 160-wide pipelined tile: NT only


@pytest.mark.parametrize("op,M,N,K,ld", [("NT", 16, 13, 64, 24), ("NN", 16, 64, 13, 24), ("TN", 13, 64, 16, 24)])
@pytest.mark.parametrize("dtype", [0, 1, 2])
def test_extents_inside_a_chunk_are_asked_for(lib, op, M, N, K, ld, dtype):
    """N of NT, k of NN, M of TN: refused unless the descriptor says that the rest of the chunk may be touched, and then only
    where the rows hold it; other epilogues, deferred sums and column sums never take a ragged N."""
    from terapipe_amd import _lib as L

    def plan(ragged=1, ld=ld, **fields):
        d = L.GemmDesc()
        d.op, d.dtype, d.M, d.N, d.K, d.ragged = {"NT": L.TP_GEMM_NT, "NN": L.TP_GEMM_NN, "TN": L.TP_GEMM_TN}[op], dtype, M, N, K, ragged
        d.A = d.B = d.C = d.bias = d.colsum_acc = 4096
        d.colsum_acc = None
        d.lda = 64 if op == "NT" else ld
        d.ldb, d.ldc = 64, ld if op == "NT" else 64
        for name, value in fields.items():
            setattr(d, name, value)
        return lib.tp_gemm_plan(ctypes.byref(d), None, None)

    assert plan() == 0 and plan(ragged=0) == 2          # TP_ERR_UNSUPPORTED
    assert plan(ld=13) == 2                             # rows that do not hold the chunk
    if op == "NT":
        assert plan(epilogue=L.TP_EPI_BIAS) == plan(defer_reduce=1) == plan(colsum_acc=4096) == 2


def test_few_large_tiles_on_a_long_k():
    """48 to 63 tiles of 256 x 256: split to one round from k = 12288 on, the estimate's choice below."""
    for M, N, splits in ((2048, 1792, 4), (1536, 2048, 5), (2000, 1600, 4)):
        assert plan("NN", M, N, 12288) == plan("NT", M, N, 12288) == (44, splits)
        assert plan("NN", M, N, 12224)[0] != 44
