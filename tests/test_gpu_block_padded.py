"""16-bit blocks whose inner width is not a multiple of 8 (laid out with padded halves, weights packed, gradients
unpacked: csrc/block_any.hip) against the float64 block oracle: gate widths 2, 6, 10, 50 and 132 + 2, even and odd extents,
and the small tensors that run unpadded."""
import pytest
import torch

from test_gpu_block import _block_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dim,k,shape", [
    (8, 17, (2, 60, 60, 8)), (24, 9, (3, 33, 40, 24)), (40, 15, (4, 13, 13, 40)), (88, 13, (2, 28, 32, 88)),
    (200, 5, (1, 57, 61, 200)), (264, 7, (2, 20, 24, 264)), (536, 3, (1, 7, 9, 536)), (40, 3, (2, 9, 8, 40)),
])
def test_padded_inner_channels(oracle, dtype, dim, k, shape):
    _block_case(oracle, dim, k, shape, dtype)
