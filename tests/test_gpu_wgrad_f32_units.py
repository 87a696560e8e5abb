"""fp32 weight gradients whose workgroups take several units (images, row bands, column tiles) as one stream
(csrc/dwconv_wgrad_f32t.h), with an odd and an even number of ticks, a last chunk of fewer units, images that stand beside
others in a tile, and totals taken more often than once a unit; against float64."""
import pytest
import torch

from parity import assert_close, randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,k", [
    ((530, 12, 13, 8), 9),     # three units a workgroup, the last chunk short; several images in a tile
    ((9, 13, 30, 520), 13),    # 65 slices of channels, three chunks of three images
    ((7, 35, 61, 300), 15),    # two column tiles an image, several chunks of both
    ((2, 70, 25, 16), 17),     # bands of one image, two products a position
    ((1, 5, 90, 12), 11),      # fewer rows than the filter
    ((1, 90, 8, 16), 15),      # a workgroup's last rows end inside an image, and three of a tile's four images are missing
    ((3, 120, 20, 8), 13),     # ... the second of two
])
def test_several_units_in_a_workgroup(oracle, shape, k):
    from pyramidconvblock_amd.dwconv import dwconv_wgrad

    B, H, W, C = shape
    gen = torch.Generator().manual_seed(k + C)
    x, g = randn(gen, B, H, W, C), randn(gen, B, H, W, C)
    dw = dwconv_wgrad(x.cuda(), g.cuda(), (k, k, C), (1, 1), (k // 2, k // 2), (1, 1))
    assert_close(dw, oracle.dwconv_wgrad(x.double().numpy(), g.double().numpy(), (k, k), 1, k // 2, 1), torch.float32, "dw")
