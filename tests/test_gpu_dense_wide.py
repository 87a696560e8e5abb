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
    """Remainders of 4 in both widths, ranges of rows that end within a stage, and many of them."""
    _layers(torch.float32, K, NO, N, P)


# (a weight gradient's tiles are its output's width by its input's)
@pytest.mark.parametrize("K,NO,N", [(448, 780, 848), (448, 780, 849), (4, 968, 5951), (28, 1048, 6829), (968, 4, 5951), (1048, 28, 6829)])
def test_fp32_weight_gradients_in_larger_tiles(K, NO, N):
    """128 x 128 and 128 x 64 results, where they are estimated to end clearly before 64 x 64 (the last two stay there): remainders of 4 and of
    a stage."""
    _layers(torch.float32, K, NO, N, N)


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


@pytest.mark.parametrize("dtype,dim,shape", [(torch.bfloat16, 400, (3, 57, 61, 400)), (torch.bfloat16, 1048, (1, 64, 67, 1048)), (torch.bfloat16, 200, (11, 51, 50, 200)),
                                             (torch.float32, 352, (6, 15, 15, 352)), (torch.float32, 872, (3, 21, 20, 872)), (torch.float32, 384, (3, 12, 15, 384))])
def test_row_ranges_that_make_room(oracle, dtype, dim, shape):
    """Row ranges that are fewer than a weight gradient by itself would have: launches of both products that the chip holds at once (400; 352, 384 and 872), and
    longer ones (200; 1048, one of its layers)."""
    _block_case(oracle, dim, 3, shape, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K,NO", [(264, 136), (320, 200), (256, 384)])
def test_dense_wide_columns_of_192(dtype, K, NO):
    """Tiles of 128 x 192: rows enough for one round of them to save one of the narrower ones, remainders in both."""
    _layers(dtype, K, NO, 257 * 128 + 5, 257 * 128 + 5)


@pytest.mark.parametrize("K,NO,N,P", [(196, 196, 13100, 13100), (516, 200, 7001, 700), (200, 516, 7001, 7001), (1028, 260, 2000, 63), (704, 352, 10816, 10816),
                                      (192, 192, 13564, 6782), (260, 1028, 2000, 2000), (768, 512, 2048, 2048), (768, 512, 2049, 2049)])
def test_large_fp32_layers(K, NO, N, P):
    """Large fp32 products: remainders of 4 results and inner values, an odd number of stages, ranges of rows, and either side of 256
    tiles; no further from float64 than fp32 products and sums of that length are (their partial sums random: sqrt(K) roundings)."""
    from pyramidconvblock_amd import ops

    _layers(torch.float32, K, NO, N, P)
    gen = torch.Generator().manual_seed(K)
    x, w = randn(gen, N, K), randn(gen, NO, K)
    y = ops.dense_forward(x.cuda(), w.cuda())
    want = x.double() @ w.double().t()
    assert float((y.double().cpu() - want).norm() / want.norm()) <= 2.0 ** -24 * K ** 0.5
    dw = ops.dense_wgrad(y, x.cuda())
    want = y.double().cpu().t() @ x.double()
    assert float((dw.double().cpu() - want).norm() / want.norm()) <= 2.0 ** -24 * N ** 0.5


def test_fp32_values_that_are_not_finite():
    """Infinities of a sign, NaN, and values near fp32's largest give what fp32 arithmetic gives; the other results are as without them."""
    from pyramidconvblock_amd import ops

    K, NO, N = 260, 256, 8000
    gen = torch.Generator().manual_seed(1)
    x, w, g = randn(gen, N, K), randn(gen, NO, K), randn(gen, N, NO)
    clean = ops.dense_forward(x.cuda(), w.cuda()).cpu()
    dclean = ops.dense_wgrad(g.cuda(), x.cuda()).cpu()
    xp = x.clone()
    xp[5, 7], xp[300, 9], xp[4000, 0] = float("inf"), float("nan"), -float("inf")
    xp[700, 11] = 3.4e38
    y = ops.dense_forward(xp.cuda(), (w * 1e-3).cuda()).cpu()
    want = xp.double() @ (w * 1e-3).double().t()
    for r in (5, 4000):
        assert torch.equal(y[r].double(), want[r])   # infinities of the weights' signs
    assert torch.isnan(y[300]).all()
    assert torch.isfinite(y[700]).all() and float(((y[700].double() - want[700]) / want[700].abs().max()).abs().max()) < 1e-6
    others = torch.ones(N, dtype=torch.bool)
    others[[5, 300, 700, 4000]] = False
    assert torch.isfinite(y[others]).all() and float((y[others].double() - want[others]).norm() / want[others].norm()) < 1e-6
    dw = ops.dense_wgrad(g.cuda(), xp.cuda()).cpu()
    for c, r in ((7, 5), (0, 4000)):
        assert torch.equal(dw[:, c].double(), (g[r].double() * xp[r, c].double()))
    assert torch.isnan(dw[:, 9]).all()
    cols = torch.ones(K, dtype=torch.bool)
    cols[[0, 7, 9, 11]] = False
    assert float((dw[:, cols] - dclean[:, cols]).norm() / dclean.norm()) < 1e-6
    wp = w.clone()
    wp[3, 4] = float("inf")
    y = ops.dense_forward(x.cuda(), wp.cuda()).cpu()
    assert torch.equal(y[:, 3].double(), x[:, 4].double() * float("inf"))
    keep = torch.ones(NO, dtype=torch.bool)
    keep[3] = False
    assert float((y[:, keep] - clean[:, keep]).norm() / clean.norm()) < 1e-6


@pytest.mark.parametrize("K", [256, 260])   # (weight gradients up to 256 wide run dense_any.hip)
def test_fp32_values_whose_products_overflow(K):
    """Infinities, and no NaN."""
    from pyramidconvblock_amd import ops

    gen = torch.Generator().manual_seed(3)
    x, w, g = randn(gen, 8000, K), randn(gen, 256, K), randn(gen, 8000, 256)
    clean = ops.dense_forward(x.cuda(), w.cuda()).cpu()
    xp, wp = x.clone(), w.clone()
    xp[5], wp[7] = (x[5].abs() + 1) * 1e23, (w[7].abs() + 1) * 1e23
    y = ops.dense_forward(xp.cuda(), wp.cuda()).cpu()
    assert y[5, 7] == float("inf")
    assert torch.isfinite(y[5, :7]).all() and torch.isfinite(y[:5, 7]).all()
    y[5], y[:, 7] = clean[5], clean[:, 7]
    assert float((y - clean).norm() / clean.norm()) < 1e-6
    xc, gc = x.clone(), g.clone()
    xc[:, 9], gc[:, 11] = (x[:, 9].abs() + 1) * 1e23, -(g[:, 11].abs() + 1) * 1e23
    dw = ops.dense_wgrad(gc.cuda(), xc.cuda()).cpu()
    assert dw[11, 9] == -float("inf") and int(torch.isfinite(dw).logical_not().sum()) == 1


@pytest.mark.parametrize("K", [256, 260])
@pytest.mark.parametrize("scale", [1e-29, 1e-34, 1e-37])
def test_fp32_values_near_the_smallest(scale, K):
    """No less precise than others."""
    from pyramidconvblock_amd import ops

    gen = torch.Generator().manual_seed(2)
    x, w = randn(gen, 8000, K), randn(gen, 256, K) * 1e4
    x[:1000] *= scale   # (beside rows of ordinary values, in tiles of their own and in one with them)
    y = ops.dense_forward(x.cuda(), w.cuda()).cpu().double()
    want = x.double() @ w.double().t()
    for rows in (slice(0, 1000), slice(1000, None)):
        assert float((y[rows] - want[rows]).norm() / want[rows].norm()) <= 2.0 ** -24 * 16
    g = randn(gen, 8000, 256) * scale
    dw = ops.dense_wgrad(g.cuda(), x[1000:].repeat(2, 1)[:8000].cuda()).cpu().double()
    want = g.double().t() @ x[1000:].repeat(2, 1)[:8000].double()
    assert float((dw - want).norm() / want.norm()) <= 2.0 ** -24 * 8000 ** 0.5


@pytest.mark.parametrize("dim,shape", [(400, (3, 47, 45, 400)), (712, (1, 50, 41, 712))])
def test_large_fp32_products_of_a_block(oracle, dim, shape):
    """Both products of a layer's backward, in one launch."""
    _block_case(oracle, dim, 3, shape, torch.float32)


def test_fp32_results_of_one_term_are_rounded_once():
    """A sum of zeros and one product is that product rounded to fp32: operands keep all their bits, and so do their products."""
    from pyramidconvblock_amd import ops

    N, K, NO = 10816, 704, 352
    gen = torch.Generator().manual_seed(4)
    at = torch.randint(0, K, (N,), generator=gen)
    v, w, g = randn(gen, N), randn(gen, NO, K), randn(gen, N, NO)
    x = torch.zeros(N, K)
    x[torch.arange(N), at] = v
    y = ops.dense_forward(x.cuda(), w.cuda()).cpu()
    assert torch.equal(y, v[:, None] * w.t()[at])
    dx = ops.dense_forward(x.cuda(), w.t().contiguous().cuda(), w_kmajor=True).cpu()
    assert torch.equal(dx, y)
    rows = torch.randint(0, N, (K,), generator=gen)
    x = torch.zeros(N, K)
    x[rows, torch.arange(K)] = v[:K]
    dw = ops.dense_wgrad(g.cuda(), x.cuda()).cpu()
    assert torch.equal(dw, (g[rows] * v[:K, None]).t())


def test_fp32_small_values_beside_ordinary_ones():
    """A column near fp32's smallest values among ordinary ones, and small values that meet large ones: as precise as the others."""
    from pyramidconvblock_amd import ops

    N, K, NO = 10816, 704, 352
    gen = torch.Generator().manual_seed(5)
    x, g, w = randn(gen, N, K), randn(gen, N, NO), randn(gen, NO, K)
    x[:, 5] *= 1e-36
    dw = ops.dense_wgrad(g.cuda(), x.cuda()).cpu().double()
    want = g.double().t() @ x.double()
    assert float((dw[:, 5] - want[:, 5]).norm() / want[:, 5].norm()) <= 2.0 ** -24 * N ** 0.5
    w[:, :] = 0
    w[:, 5] = 1e30
    y = ops.dense_forward(x.cuda(), w.cuda()).cpu().double()
    want = x.double() @ w.double().t()
    assert float((y - want).norm() / want.norm()) <= 2.0 ** -24


def test_fp32_products_take_as_long_whatever_the_values():
    """A NaN in every tile does not slow a product down (a bound far above what timings scatter by: a fifth at most)."""
    from pyramidconvblock_amd import ops

    x, w = torch.randn(10816, 704, device="cuda"), torch.randn(352, 704, device="cuda")
    bad = x.clone()
    bad[::64, 3] = float("nan")

    def ms(a):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        ops.dense_forward(a, w), ops.dense_wgrad(a, a)
        start.record()
        for _ in range(20):
            ops.dense_forward(a, w), ops.dense_wgrad(a, a)
        end.record()
        end.synchronize()
        return start.elapsed_time(end)

    assert min(ms(bad) for _ in range(3)) < 4 * min(ms(x) for _ in range(3))


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
