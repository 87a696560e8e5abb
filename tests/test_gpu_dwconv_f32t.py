"""The fp32 convolutions on the fp32 matrix cores (csrc/dwconv_f32t.h, csrc/dwconv_wgrad_f32t.h) against float64, at the edges
of their tiles (columns, images side by side, row bands, channel slices) and with pooled gradients of any ratio."""
import pytest
import torch

from parity import assert_close, randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [3, 5, 7, 9, 11, 13, 15, 17])
@pytest.mark.parametrize("shape,hw", [((1, 5, 1, 4), (2, 1)), ((5, 9, 8, 12), (4, 4)), ((3, 12, 33, 20), (6, 16)), ((2, 37, 64, 8), (37, 30)),
                                      ((3, 21, 24, 16), (10, 12)), ((1, 50, 65, 36), (25, 32)), ((9, 18, 16, 8), (9, 8))])
def test_f32_matrix_core_convolutions(oracle, k, shape, hw):
    from pyramidconvblock_amd.dwconv import dwconv_dgrad, dwconv_forward, dwconv_wgrad

    B, H, W, C = shape
    gen = torch.Generator().manual_seed(k * H + W)
    w = randn(gen, k, k, C) / k
    for pad in (k // 2, min(k - 1, k // 2 + 2)):
        x, gp = randn(gen, B, H, W, C), randn(gen, B, *hw, C)
        geo = ((1, 1), (pad, pad), (1, 1))
        y = dwconv_forward(x.cuda(), w.cuda(), *geo)
        xn, wn = x.double().numpy(), w.double().numpy()
        assert_close(y, oracle.dwconv_fwd(xn, wn, 1, pad, 1), torch.float32, "y")
        g = randn(gen, *y.shape)
        gn = g.double().numpy()
        dx_ref = oracle.dwconv_dgrad(gn, wn, (H, W), 1, pad, 1)
        assert_close(dwconv_dgrad(g.cuda(), w.cuda(), x.shape, *geo), dx_ref, torch.float32, "dx")
        dx = dwconv_dgrad(g.cuda(), w.cuda(), x.shape, *geo, pooled_grad=gp.cuda())
        assert_close(dx, dx_ref + oracle.avgpool_bwd(gp.double().numpy(), (H, W)), torch.float32, "dx + pooled")
        dw = dwconv_wgrad(x.cuda(), g.cuda(), (k, k, C), *geo)
        assert_close(dw, oracle.dwconv_wgrad(xn, gn, (k, k), 1, pad, 1), torch.float32, "dw")


@pytest.mark.parametrize("k", [3, 9, 13, 15, 17])
@pytest.mark.parametrize("shape,hw", [((2, 32, 32, 32), (16, 16)), ((3, 57, 61, 100), (28, 30)), ((5, 13, 18, 12), (6, 9)), ((9, 40, 56, 8), (20, 28))])
def test_weight_gradients_of_two_scales_in_one_launch(k, shape, hw):
    """The pair launch's results are bitwise the single launches'."""
    from pyramidconvblock_amd.dwconv import dwconv_wgrad, dwconv_wgrad_pair

    B, H, W, C = shape
    gen = torch.Generator().manual_seed(k + W)
    x0, g0 = (randn(gen, B, H, W, C).cuda() for _ in range(2))
    x1, g1 = (randn(gen, B, *hw, C).cuda() for _ in range(2))
    geo = ((1, 1), (k // 2, k // 2), (1, 1))
    d0, d1 = dwconv_wgrad_pair(x0, g0, x1, g1, (k, k, C))
    assert torch.equal(d0, dwconv_wgrad(x0, g0, (k, k, C), *geo)) and torch.equal(d1, dwconv_wgrad(x1, g1, (k, k, C), *geo))


@pytest.mark.parametrize("k", [3, 9, 17])
@pytest.mark.parametrize("shape", [(1, 2, 64, 4), (1, 6, 8, 12), (3, 10, 30, 8), (1, 50, 16, 20)])
def test_pooled_gradient_below_the_last_row(oracle, k, shape):
    """Exact halves whose last patch row, and those requested after it, lie below the pooled gradient's last row."""
    from pyramidconvblock_amd.dwconv import dwconv_dgrad

    B, H, W, C = shape
    gen = torch.Generator().manual_seed(k + H)
    g, gp, w = randn(gen, *shape), randn(gen, B, H // 2, W // 2, C), randn(gen, k, k, C) / k
    dx = dwconv_dgrad(g.cuda(), w.cuda(), shape, (1, 1), (k // 2, k // 2), (1, 1), pooled_grad=gp.cuda())
    want = oracle.dwconv_dgrad(g.double().numpy(), w.double().numpy(), (H, W), 1, k // 2, 1)
    assert_close(dx, want + oracle.avgpool_bwd(gp.double().numpy(), (H, W)), torch.float32)
