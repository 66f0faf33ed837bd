"""LayerNorm rows alone (no parameter gradients beside) at the edges of the rule that says how many chunks a thread holds: row
counts around its steps, rows whose last chunk falls short of a thread's share, one row, the widest row; against fp64."""
import pytest
import torch

from tests.util import assert_close

DEV = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=str)
@pytest.mark.parametrize("M,chunks", [(1, 1), (3, 65), (2047, 127), (2048, 128), (2049, 203), (2048, 511), (511, 512), (512, 513),
                                      (1023, 640), (1024, 769), (1025, 512), (5, 4096), (1024, 4095),
                                      (7, 257), (300, 448), (40, 769), (2048, 1536), (2048, 1537)], ids=str)
def test_rows(M, chunks, dtype):
    from terapipe_amd import ops
    E = chunks * (4 if dtype == torch.float32 else 8)
    g = torch.Generator(device=DEV).manual_seed(M + chunks)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    x, dy, res = (rnd(M, E).to(dtype) for _ in range(3))
    gamma, beta = (1 + 0.2 * rnd(E)).to(dtype), rnd(E).to(dtype)
    y, mean, rstd = ops.layernorm_fwd(x, gamma, beta)
    xd = x.double().requires_grad_()
    want = torch.nn.functional.layer_norm(xd, (E,), gamma.double(), beta.double())
    want.backward(dy.double())
    assert_close(y, want.detach(), dtype, "y")
    assert_close(ops.layernorm_bwd(dy, x, mean, rstd, gamma, None, None, None), xd.grad, dtype, "dx")
    assert_close(ops.layernorm_bwd(dy, x, mean, rstd, gamma, res, None, None), xd.grad + res.double(), dtype, "dx + residual")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=str)
@pytest.mark.parametrize("splits", [2, 3, 4, 5, 8, 9, 31, 32])
def test_partial_sums_are_added_in_the_order_of_the_splits(splits, dtype):
    """Rows that arrive as a split product's partial sums, forward and backward: the tensor written is, bit for bit, their sum in
    order (with bias and residual), and the rows after it are those of that tensor."""
    from terapipe_amd import ops
    M, E = 5, 328
    g = torch.Generator(device=DEV).manual_seed(splits)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    ws, bias, res, x = rnd(splits, M, E), rnd(E).to(dtype), rnd(M, E).to(dtype), rnd(M, E).to(dtype)
    gamma, beta = (1 + 0.2 * rnd(E)).to(dtype), rnd(E).to(dtype)
    total = torch.zeros(M, E, device=DEV)
    for part in ws:
        total = total + part
    h = torch.full((M, E), float("nan"), dtype=dtype, device=DEV)
    y, mean, rstd = ops.layernorm_fwd(ops.PendingReduce(ws, splits, bias, res, h), gamma, beta)
    assert torch.equal(h, ((total + bias.float()) + res.float()).to(dtype))
    for got, want in zip((y, mean, rstd), ops.layernorm_fwd(h, gamma, beta)):
        assert torch.equal(got, want)
    dy = torch.full((M, E), float("nan"), dtype=dtype, device=DEV)
    _, mean, rstd = ops.layernorm_fwd(x, gamma, beta)
    dx = ops.layernorm_bwd(ops.PendingReduce(ws, splits, None, None, dy), x, mean, rstd, gamma, res, None, None)
    assert torch.equal(dy, total.to(dtype)) and torch.equal(dx, ops.layernorm_bwd(dy, x, mean, rstd, gamma, res, None, None))
