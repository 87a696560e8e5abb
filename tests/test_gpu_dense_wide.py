"""The 128 x 128-tile dense kernels (csrc/dense_wide.hip: 16-bit layers wider than 128, fp32 layers) against float64, at the
edges of their tiles, stages and row ranges."""
import pytest
import torch

from parity import assert_close, randn
from test_gpu_block import _block_case

pytestmark = pytest.mark.gpu


def _layers(dtype, K, NO, N, P):
    from pyramidconvblock_amd import ops

    assert dtype == torch.float32 or (ops.dense_supported(K, NO, dtype) and ops.dense_supported(NO, K, dtype))
    gen = torch.Generator().manual_seed(K + NO + N)
    x, g = randn(gen, N, K).to(dtype), randn(gen, N, NO).to(dtype)
    w, b = (randn(gen, NO, K) / K ** 0.5).to(dtype), randn(gen, NO).to(dtype)
    rb = randn(gen, (N + P - 1) // P, NO)
    y = ops.dense_forward(x.cuda(), w.cuda(), bias=b.cuda(), rowbias=rb.cuda(), rows_per_image=P)
    ref = x.double() @ w.double().t() + b.double() + rb.double().repeat_interleave(P, 0)[:N]
    assert_close(y, ref.numpy(), dtype, "forward", 0.5)
    dx = ops.dense_forward(g.cuda(), w.cuda(), w_kmajor=True)
    assert_close(dx, (g.double() @ w.double()).numpy(), dtype, "input gradient", 0.5)
    dw = ops.dense_wgrad(g.cuda(), x.cuda())
    assert_close(dw, (g.double().t() @ x.double()).numpy(), dtype, "weight gradient", 0.5)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K,NO", [(136, 8), (8, 264), (200, 112), (256, 128), (520, 264), (64, 192), (1152, 576)])
@pytest.mark.parametrize("N,P", [(1, 1), (63, 7), (130, 65), (1000, 250), (4097, 4097)])
def test_dense_wide_layers(dtype, K, NO, N, P):
    _layers(dtype, K, NO, N, P)


@pytest.mark.parametrize("K,NO", [(4, 4), (132, 36), (100, 200), (128, 64), (64, 128), (260, 576)])
@pytest.mark.parametrize("N,P", [(1, 1), (63, 7), (1000, 250), (4097, 4097), (70001, 35001)])
def test_dense_wide_fp32_layers(K, NO, N, P):
    """Every tile (70001 rows: 128 high), remainders of 4 in both widths, ranges of rows that end within a stage."""
    _layers(torch.float32, K, NO, N, P)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K,NO", [(376, 136), (384, 64), (392, 72), (448, 920), (1152, 144)])
@pytest.mark.parametrize("N", [1, 65, 191, 320, 2128])
def test_few_workgroups_of_long_sums(dtype, K, NO, N):
    """Four stages in flight: sums just below and from six stages on (of three in a weight gradient's range), remainders of a stage,
    every tile."""
    _layers(dtype, K, NO, N, N)


@pytest.mark.parametrize("dim,shape", [(920, (2, 9, 8, 920)), (520, (3, 14, 13, 520)), (264, (1, 6, 5, 264))])
def test_few_workgroups_of_both_products(oracle, dim, shape):
    """The same in the launch that makes both gradients of a block's layers."""
    _block_case(oracle, dim, 3, shape, torch.float16)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K,NO", [(264, 136), (320, 200), (256, 384)])
def test_dense_wide_columns_of_192(dtype, K, NO):
    """Tiles of 128 x 192: rows enough for one round of them to save one of the narrower ones, remainders in both."""
    _layers(dtype, K, NO, 257 * 128 + 5, 257 * 128 + 5)


@pytest.mark.parametrize("dtype,N", [(torch.bfloat16, 270000), (torch.float32, 140000)])
def test_weight_gradient_of_more_than_2_gib(dtype, N):
    """A layer whose tiles alone fill the chip, over operands that one range's 32-bit offsets do not reach."""
    from pyramidconvblock_amd import ops

    M, NO = 4096, 2048
    gen = torch.Generator(device="cuda").manual_seed(6)
    a = torch.randn(N, M, generator=gen, device="cuda").to(dtype)
    b = torch.randn(N, NO, generator=gen, device="cuda").to(dtype)
    assert a.numel() * a.element_size() > 2**31
    got = ops.dense_wgrad(a, b)
    cols = torch.tensor([0, 127, 128, 2047, 4095], device="cuda")
    want = sum(a[i:i + 20000, cols].double().t() @ b[i:i + 20000].double() for i in range(0, N, 20000))
    assert_close(got[cols], want.cpu().numpy(), dtype, "dw")
