"""The measured plans of products that run beside other streams' launches (bit 24 of tp_gemm_desc.reserved): every entry of their table
is the plan with the bit, the entry of the main table without it, and other shapes ignore the bit.  Host arithmetic only."""
import ctypes
import os
import re

from terapipe_amd import _lib as L


def _plan(op, M, N, K, reserved):
    d = L.GemmDesc()
    d.op, d.dtype, d.epilogue, d.M, d.N, d.K, d.reserved = op, L.TP_F16, L.TP_EPI_STORE, M, N, K, reserved
    d.A = d.B = d.C = 4096
    d.lda, d.ldb, d.ldc = K, (K if op == L.TP_GEMM_NT else N), N
    c, n = ctypes.c_int(), ctypes.c_int()
    assert L.load().tp_gemm_plan(ctypes.byref(d), ctypes.byref(c), ctypes.byref(n)) == 0
    return c.value, n.value


def _entries(name):
    text = open(os.path.join(os.path.dirname(L.__file__), "csrc", name)).read()
    return {(getattr(L, "TP_GEMM_" + m[0]),) + tuple(int(v) for v in m[1:4]): (int(m[4]), int(m[5]))
            for m in re.findall(r"^\{TP_GEMM_(NT|NN), (\d+), (\d+), (\d+), (\d+), (\d+)\}", text, re.M)}


def test_plans_beside_other_streams():
    alone, beside = _entries("gemm_tuned.inc"), _entries("gemm_tuned_beside.inc")
    assert beside and set(beside) <= set(alone)
    for key, want in alone.items():
        assert _plan(*key, 0) == want
        assert _plan(*key, 1 << 24) == beside.get(key, want)
    for key in ((L.TP_GEMM_NT, 300, 1000, 3000), (L.TP_GEMM_NN, 2048, 4096, 4096), (L.TP_GEMM_NT, 16, 2048, 2048)):
        assert _plan(*key, 1 << 24) == _plan(*key, 0)


def test_the_benchmark_names_the_products_of_the_table():
    import bench
    assert bench.in_step_picks() == set(_entries("gemm_tuned_beside.inc"))
