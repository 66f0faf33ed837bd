"""The tiled attention kernels at head dimensions 80 and 96 (rows that do not fill a power of two of 16-byte chunks), at
the edges of their tiles: the checks of test_kernels_gpu.py against the fp64 oracle, at other shapes."""
import pytest
import torch

from tests import test_kernels_gpu as k

DTYPES = pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
pytestmark = pytest.mark.gpu


@DTYPES
@pytest.mark.parametrize("Dh", [80, 96])
@pytest.mark.parametrize("T,B,H,P,L", [
    (1, 1, 1, 0, 1), (1, 2, 3, 64, 80), (31, 1, 2, 1, 32),      # one row; one short of a block
    (33, 2, 2, 0, 40), (64, 1, 2, 63, 127), (65, 1, 1, 129, 256),
    (300, 1, 2, 0, 300), (129, 3, 2, 511, 640),                 # several blocks, the last one ragged
], ids=str)
def test_slice_forward_backward(dtype, Dh, T, B, H, P, L):
    k.test_attn_prefix_fwd_bwd(dtype, T, B, H, Dh, P, L)


@DTYPES
@pytest.mark.parametrize("B,H,Dh,L,slices", [
    (2, 2, 80, 96, [32, 32, 32]), (2, 1, 96, 64, [5, 1, 20]), (1, 3, 80, 200, [40, 7, 100, 33]),
    (1, 2, 96, 512, [128, 128, 128, 128]), (1, 2, 80, 700, [577, 123]),
], ids=str)
def test_position_indexed(dtype, B, H, Dh, L, slices):
    k.test_attn_position_indexed_and_suffix_dkdv(dtype, B, H, Dh, L, slices)


@DTYPES
@pytest.mark.parametrize("T,B,H,Dh,P,ns", [(32, 2, 3, 80, 480, 2), (40, 1, 2, 96, 200, 3), (7, 1, 2, 80, 1000, 4)], ids=str)
def test_keys_shared_by_workgroups(dtype, T, B, H, Dh, P, ns):
    k.test_attn_fwd_keys_shared_by_workgroups(dtype, T, B, H, Dh, P, ns)
