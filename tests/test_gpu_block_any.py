"""16-bit blocks whose inner width is not a multiple of 8 (laid out with padded halves, weights packed, gradients
unpacked: csrc/block_any.hip) against the float64 block oracle: gate widths 2, 6, 10, 50 and 132 + 2, even and odd extents,
small tensors and large ones."""
import pytest
import torch

from parity import assert_close
from test_gpu_block import _block_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dim,k,shape", [
    (8, 17, (2, 60, 60, 8)), (24, 9, (3, 33, 40, 24)), (40, 15, (4, 13, 13, 40)), (88, 13, (2, 28, 32, 88)),
    (200, 5, (1, 57, 61, 200)), (264, 7, (2, 20, 24, 264)), (536, 3, (1, 7, 9, 536)), (40, 3, (2, 9, 8, 40)),
    (8, 3, (1, 2, 2, 8)), (24, 17, (1, 7, 7, 24)), (56, 5, (2, 3, 16, 56)), (136, 9, (1, 2, 31, 136)), (248, 13, (1, 7, 8, 248)),
])
def test_padded_inner_channels(oracle, dtype, dim, k, shape):
    _block_case(oracle, dim, k, shape, dtype)


@pytest.mark.parametrize("dim,inter,k,shape,shift", [
    # conv_up on tiles of whole images with their sums (a width that fills the tiles, and one that does not), on others, on
    # wide tiles of 64 and 128 results, and on weights that it does not read in place (8 bytes off the alignment)
    (128, 124, 5, (2, 32, 32), 0), (72, 36, 7, (2, 32, 32), 0), (104, 52, 7, (1, 30, 34), 0), (136, 68, 5, (2, 32, 32), 0),
    (264, 132, 3, (1, 9, 11), 0), (392, 196, 3, (1, 7, 12), 0), (104, 52, 7, (1, 30, 34), 4), (264, 132, 3, (1, 9, 11), 4),
])
def test_weights_read_as_given_and_packed_beside_the_pool(oracle, dim, inter, k, shape, shift):
    """Padded halves: conv_up skips the rows that its weights do not have, the pool's launch packs all four."""
    import pyramid_dwconv

    dtype = torch.bfloat16
    torch.manual_seed(3)
    m = pyramid_dwconv.ConvBlock(dim=dim, kernel_size=k, inter_ratio=inter / dim).to(dtype)
    x, g = (torch.randn(*shape, dim).to(dtype) for _ in range(2))
    params = {n: p.detach().double().numpy() for n, p in m.state_dict().items()}
    yo, cache = oracle.convblock_fwd(x.double().numpy(), params)
    dxo, go = oracle.convblock_bwd(cache, g.double().numpy())
    m = m.cuda()
    w = m.conv_up.weight
    w.data = torch.cat([w.data.new_zeros(shift), w.data.flatten()])[shift:].view_as(w)
    xd = x.cuda().requires_grad_()
    y = m(xd)
    assert_close(y, yo, dtype, "y")
    torch.autograd.backward(y, g.cuda())
    assert_close(xd.grad, dxo, dtype, "dx")
    for n, p in m.named_parameters():
        assert_close(p.grad, go[n], dtype, "grad " + n)


@pytest.mark.parametrize("dtype,dim,k,shape", [
    (torch.bfloat16, 16, 5, (5, 11, 13, 16)), (torch.float16, 72, 3, (2, 90, 90, 72)), (torch.bfloat16, 1032, 3, (1, 7, 9, 1032)),
    (torch.float32, 36, 5, (3, 17, 12, 36)), (torch.float32, 252, 3, (40, 9, 8, 252)), (torch.float16, 256, 3, (70, 6, 6, 256)),
    # the forward with everything in flight: a last slice of 4, 8 and 16 features, one partial and many, more columns than twice the threads
    (torch.float32, 260, 3, (3, 9, 8, 260)), (torch.float16, 264, 3, (2, 30, 33, 264)), (torch.bfloat16, 272, 3, (1, 41, 64, 272)),
    (torch.bfloat16, 2056, 3, (2, 5, 4, 2056)), (torch.float32, 2080, 3, (1, 4, 6, 2080)),
    # four images to a workgroup of its backward: a rest of one and of two, sums of one and of several ranges
    (torch.bfloat16, 264, 3, (41, 6, 6, 264)), (torch.float16, 136, 3, (66, 5, 6, 136)), (torch.bfloat16, 520, 3, (22, 16, 18, 520)),
])
def test_mean_branch_of_any_width(oracle, dtype, dim, k, shape):
    """The mean branch riding in the pool's and the gates' launches (csrc/mean_any.h): widths of less than one, of several
    and of more than 256 vectors of four sums, one and many ranges of positions, batches beyond its plan's."""
    _block_case(oracle, dim, k, shape, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dim,k,shape", [
    (16, 13, (3, 9, 70, 16)), (32, 17, (2, 33, 31, 32)), (48, 3, (5, 65, 33, 48)), (144, 9, (1, 12, 66, 144)), (80, 15, (3, 14, 32, 80)),
    (176, 11, (9, 8, 8, 176)),
])
def test_convolutions_of_any_two_scales(oracle, dtype, dim, k, shape):
    """Both scales' convolutions in one launch, forward and backward (csrc/dwconv_fwd2.h, dwconv_bwd3.h): wide and narrow tiles
    of either scale, odd batches in two-image tiles, pooled extents that are exact halves and not, a last slice of 8 channels."""
    _block_case(oracle, dim, k, shape, dtype)


@pytest.mark.parametrize("k", [3, 9, 13, 17])
@pytest.mark.parametrize("dim,shape", [(16, (1, 12, 64, 16)), (24, (3, 33, 31, 24)), (8, (5, 17, 16, 8)), (40, (2, 9, 130, 40))])
def test_fp32_convolutions_of_two_scales(oracle, k, dim, shape):
    """Both scales' fp32 convolutions in one launch (csrc/dwconv_f32t.h): tiles of one, two and four images, two column tiles,
    odd batches and extents, slices of 4 channels."""
    _block_case(oracle, dim, k, shape, torch.float32)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(2, 2, 2, 16), (1, 2, 3, 64), (5, 4, 4, 32), (1, 6, 6, 8), (64, 4, 8, 64), (3, 8, 8, 136)])
def test_sums_of_x_in_the_result_or_behind_the_saved(oracle, dtype, shape):
    """The forward's sums of x, in y until it is written, or (images of a few pixels) in the buffer of the saved tensors."""
    _block_case(oracle, shape[3], 3, shape, dtype)


@pytest.mark.parametrize("dtype,dim,k,shape", [
    # pairs of image rows of one quad and of many, quads that end within a tile of 64 or 128 rows and an image that ends within one
    (torch.float32, 64, 3, (3, 2, 2, 64)), (torch.float32, 132, 3, (5, 6, 10, 132)), (torch.float32, 200, 5, (2, 34, 2, 200)),
    (torch.float32, 32, 3, (1, 2, 66, 32)), (torch.bfloat16, 144, 3, (3, 2, 2, 144)), (torch.float16, 264, 3, (5, 6, 10, 264)),
    (torch.bfloat16, 400, 3, (2, 34, 2, 400)), (torch.float16, 640, 3, (1, 2, 66, 640)),
    # four stages in flight; packed weights; tiles of 128 rows
    (torch.bfloat16, 528, 3, (3, 14, 14, 528)), (torch.float16, 136, 3, (2, 10, 6, 136)), (torch.bfloat16, 424, 3, (3, 4, 8, 424)),
])
def test_pool_in_the_first_layers_store(oracle, dtype, dim, k, shape):
    """Wide and fp32 blocks on exact halves: conv_up's rows by 2 x 2 quads, their mean in its store (csrc/dense_wide.hip)."""
    _block_case(oracle, dim, k, shape, dtype)


@pytest.mark.parametrize("dtype,dim,shape", [
    (torch.bfloat16, 288, (11, 56, 56, 288)), (torch.float16, 576, (7, 70, 50, 576)), (torch.float16, 1152, (4, 64, 64, 1152)),
    (torch.bfloat16, 808, (4, 66, 62, 808)), (torch.float32, 128, (12, 56, 54, 128)),
    # odd extents: the sums of the output's gradient only
    (torch.bfloat16, 304, (3, 71, 67, 304)), (torch.float32, 264, (2, 67, 65, 264)), (torch.float16, 1040, (1, 65, 63, 1040)),
])
def test_pool_and_sums_beside_large_products(monkeypatch, dtype, dim, shape):
    """The same on tiles of 128 x 128 and 128 x 192 results, with padded halves too, and the sums of the output's gradient beside conv_out's gradients,
    against the separate launches: the same roundings, but for sums of x and of the output's gradient over other ranges (a rounding of the mean and what follows from it)."""
    import pyramid_dwconv
    from pyramidconvblock_amd import conv_block

    torch.manual_seed(1)
    m = pyramid_dwconv.ConvBlock(dim=dim, kernel_size=3).to(dtype).cuda()
    x, g = (torch.randn(*shape, device="cuda").to(dtype) for _ in range(2))

    def step():
        xd = x.clone().requires_grad_()
        m.zero_grad(set_to_none=True)
        y = m(xd)
        torch.autograd.backward(y, g)
        return [y.detach(), xd.grad, *[p.grad for p in m.parameters()]]

    got = step()
    monkeypatch.setattr(conv_block, "FORCE_STEPWISE", True)
    for a, b in zip(got, step()):
        assert_close(a, b.double().cpu().numpy(), dtype, "block", 0.5)


@pytest.mark.parametrize("k,dim,shape", [
    # the pooled scale's input gradient behind the weight gradients and in front (448 to 512 of their workgroups), in tiles of one, two and four images
    (3, 16, (2, 24, 26, 16)), (5, 24, (3, 26, 30, 24)), (7, 40, (1, 31, 29, 40)), (11, 72, (2, 40, 26, 72)), (13, 8, (5, 26, 27, 8)), (13, 64, (2, 24, 130, 64)),
    (9, 128, (3, 30, 30, 128)), (3, 128, (16, 30, 26, 128)), (3, 128, (16, 48, 26, 128)),
])
def test_fp32_half_scale_beside_the_weight_gradients(oracle, k, dim, shape):
    """Both weight gradients and the pooled scale's input gradient as one launch (csrc/dwconv_wgrad_f32t.h)."""
    _block_case(oracle, dim, k, shape, torch.float32)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("k", [3, 5, 7, 9, 11, 15, 17])
@pytest.mark.parametrize("shape,second", [
    # one bin a pixel and two, on either axis; runs over images of fewer rows than a step and of many; narrow and wide tiles; a last slice
    # of 8 channels; every pixel a bin of its own on one axis
    ((3, 57, 61, 48), 0.5), ((5, 7, 9, 16), 0.5), ((33, 15, 15, 32), 0.5), ((2, 3, 70, 48), 0.5), ((3, 31, 32, 16), 1 / 3), ((2, 20, 23, 32), 0.75),
    ((2, 9, 66, 16), 0.95),
])
def test_pooled_gradient_of_any_ratio_in_the_store(oracle, dtype, k, shape, second):
    """16-bit blocks whose pooled extents are no exact halves: the pool's gradient is added where the full scale's input gradient is stored
    (csrc/dwconv_tz.h, MODE 16; filter 11: by the launch behind it)."""
    import pyramid_dwconv

    torch.manual_seed(2)
    dim = shape[3]
    m = pyramid_dwconv.ConvBlock(dim=dim, kernel_size=k, scales=(1.0, second)).to(dtype)
    x, g = (torch.randn(*shape).to(dtype) for _ in range(2))
    params = {n: p.detach().double().numpy() for n, p in m.state_dict().items()}
    yo, cache = oracle.convblock_fwd(x.double().numpy(), params, scales=(1.0, second))
    dxo, go = oracle.convblock_bwd(cache, g.double().numpy())
    m = m.cuda()
    xd = x.cuda().requires_grad_()
    y = m(xd)
    assert_close(y, yo, dtype, "y")
    torch.autograd.backward(y, g.cuda())
    assert_close(xd.grad, dxo, dtype, "dx")
    for n, p in m.named_parameters():
        assert_close(p.grad, go[n], dtype, "grad " + n)


@pytest.mark.parametrize("k,shape,pooled", [
    # bins of 2 and 3 a side, of 3 and 4, of 1 and 2 on one axis with one pixel each on the other; one image and two side by side in a tile
    (9, (3, 57, 61, 200), (28, 30)), (3, (2, 111, 70, 72), (55, 35)), (17, (4, 61, 50, 104), (20, 16)), (7, (66, 15, 15, 64), (7, 7)), (5, (4, 40, 41, 168), (30, 41)),
    (15, (5, 33, 64, 96), (16, 31)),
])
def test_pooled_gradient_in_the_store_is_the_pools(k, shape, pooled):
    """The same bits as the pool's gradient added by its own launch (fp16: of a million elements, some ten would round otherwise with weights
    one rounding off)."""
    import ctypes

    from pyramidconvblock_amd import _lib

    L, dt = _lib.lib(), torch.float16
    both = L["_ZN3pdw18dwconv_bwd3_launchEPKvS1_S1_PvS1_S2_S2_S1_S1_S2_S2_iiiiiiiiP12ihipStream_tPiPKNS_7MeanJobE"]
    pool = L["_ZN3pdw18avgpool_bwd_launchEPKvPviiiiiiiiP12ihipStream_t"]
    B, H, W, C = shape
    h, w = pooled
    gen = torch.Generator(device="cuda").manual_seed(k)
    r = lambda *s: torch.randn(*s, generator=gen, device="cuda").to(dt)
    gy, x, w0, add, gy1, x1 = r(*shape), r(*shape), r(k, k, C), r(B, h, w, C), r(B, h, w, C), r(B, h, w, C)
    dw = torch.empty_like(w0)
    ws = [torch.empty(L.pdw_dwconv_wgrad_workspace_bytes(B, *e, C, k, k, 1, 1, k // 2, k // 2, 1, 1, _lib.dtype_code(dt)) // 4 + 1, device="cuda")
          for e in ((H, W), (h, w))]
    at, s = lambda t: ctypes.c_void_p(t.data_ptr() if t is not None else 0), ctypes.c_void_p(_lib.stream_ptr(x.device))
    dx = []
    for a in (add, None):
        dx.append(torch.full_like(x, float("nan")))
        rc = both(at(gy), at(w0), at(a), at(dx[-1]), at(x), at(dw), at(ws[0]), at(x1), at(gy1), at(dw), at(ws[1]), B, H, W, h, w, C, k,
                  _lib.dtype_code(dt), s, at(None), at(None))
        assert rc == 0
    assert pool(at(add), at(dx[1]), B, H, W, C, h, w, 1, _lib.dtype_code(dt), s) == 0
    assert bool(dx[1].isfinite().all()) and torch.equal(*dx)


def test_pooled_gradient_behind_the_store(oracle):
    """Odd extents where the pooled gradient is better added by a launch of its own (16 steps a run that ends last)."""
    _block_case(oracle, 664, 9, (54, 11, 8, 664), torch.bfloat16)


def test_error_of_riding_sums():
    """The sums of a large output gradient (100352 rows) in fp32 are no further off than by 512 workgroups: their chains of 25 values a thread, 8 threads, 16 ranges
    and 32 images make 2.53e-8 * sqrt(4.3e6 / 100352) in the 2-norm (a rounding's mean square for values spread over an octave, times the variances of all sums
    that are rounded); one after the other in 6 longer ranges, 1.9e-7."""
    import pyramid_dwconv

    err = []
    for seed in range(4):
        torch.manual_seed(seed)
        m = pyramid_dwconv.ConvBlock(dim=128, kernel_size=3).cuda()
        x, g = (torch.randn(32, 56, 56, 128, device="cuda") for _ in range(2))
        torch.autograd.backward(m(x), g)
        want = g.double().sum((0, 1, 2))
        for p in (p for n, p in m.named_parameters() if n.endswith("bias")):
            err.append(float((p.grad.double() - want).norm() / want.norm()))
    assert len(err) == 8 and sum(err) / 8 <= 1.66e-7, err


@pytest.mark.parametrize("k,shape", [
    # behind the weight gradients' workgroups and in front of them (448 to 512 of those), tiles of one, two and four images
    (9, (3, 30, 30, 64)), (3, (16, 30, 26, 64)), (5, (16, 40, 64, 32)), (11, (2, 40, 64, 32)), (11, (16, 30, 64, 32)), (13, (2, 24, 130, 32)), (13, (16, 30, 64, 32)),
    (15, (2, 60, 64, 32)), (15, (3, 57, 61, 100)), (15, (16, 30, 64, 32)), (17, (2, 60, 64, 32)), (17, (16, 30, 64, 32)),
])
def test_fp32_half_scale_in_the_weight_gradients_launch(k, shape):
    """That launch by its name (csrc/dwconv_wgrad_f32t.h), which has to take the case: the pooled scale's input gradient and both weight gradients
    against float64."""
    import ctypes

    import torch.nn.functional as F

    from pyramidconvblock_amd import _lib

    L, (B, H, W, C) = _lib.lib(), shape
    joint = L["_ZN3pdw29dwconv_wgrad_f32t_pair_launchEPKvS1_PvS2_iiS1_S1_S2_S2_iiiiiiP12ihipStream_tPKNS_7MeanJobES1_S2_"]
    gen = torch.Generator(device="cuda").manual_seed(k)
    r = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    ext = ((H, W), (H // 2, W // 2))
    x, gy, w1 = [r(B, *e, C) for e in ext], [r(B, *e, C) for e in ext], r(k, k, C) / k
    dw, dx1 = [torch.empty(k, k, C, device="cuda") for _ in ext], torch.empty_like(x[1])
    ws = [torch.empty(L.pdw_dwconv_wgrad_workspace_bytes(B, *e, C, k, k, 1, 1, k // 2, k // 2, 1, 1, 0) // 4 + 1, device="cuda") for e in ext]
    at = lambda t: ctypes.c_void_p(t.data_ptr())
    none, s = ctypes.c_void_p(0), ctypes.c_void_p(_lib.stream_ptr(dx1.device))
    assert _lib.dtype_code(torch.float32) == 0
    assert joint(at(x[0]), at(gy[0]), at(dw[0]), at(ws[0]), *ext[0], at(x[1]), at(gy[1]), at(dw[1]), at(ws[1]), *ext[1], B, C, k, k // 2, s, none,
                 at(w1), at(dx1)) == 0
    nchw = lambda t: t.double().cpu().permute(0, 3, 1, 2)
    oihw = lambda t: t.double().cpu().permute(2, 0, 1).unsqueeze(1)
    for i in range(2):
        xr, wr = nchw(x[i]).requires_grad_(), oihw(w1).requires_grad_()
        F.conv2d(xr, wr, padding=k // 2, groups=C).backward(nchw(gy[i]))
        assert_close(dw[i], wr.grad.squeeze(1).permute(1, 2, 0).numpy(), torch.float32, "grad w%d" % i)
    assert_close(dx1, xr.grad.permute(0, 2, 3, 1).numpy(), torch.float32, "dx")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape,half,padded", [
    # tiles of 64 x 64 in two stages and in four, 64 x 128, 128 x 64, 128 x 128, 128 x 192; an image that ends within a tile, tiles past the last row
    ((2, 20, 22, 264), 32, 32), ((2, 20, 22, 400), 32, 32), ((3, 14, 18, 520), 72, 72), ((11, 56, 56, 136), 32, 32), ((4, 66, 62, 264), 72, 72), ((6, 62, 60, 256), 192, 192),
    # the same with padded halves, whose weights are packed beside
    ((2, 20, 22, 264), 30, 32), ((2, 20, 22, 400), 27, 32), ((3, 14, 18, 520), 66, 72), ((11, 56, 56, 136), 30, 32), ((4, 66, 62, 264), 66, 72), ((6, 62, 60, 256), 190, 192),
])
def test_first_layer_with_pool_and_sums(dtype, shape, half, padded):
    """The first layer's launch by its name (csrc/dense_wide.hip) in every tile: its result and the sums of its input against float64, the pool and the packed weights
    to the bit."""
    import ctypes

    from pyramidconvblock_amd import _lib

    class Sums(ctypes.Structure):   # ColsumJob of csrc/mean_any.h
        _fields_ = [("x", ctypes.c_void_p), ("part", ctypes.c_void_p)] + [(n, ctypes.c_int) for n in ("B", "P", "C", "n", "len", "lanes_log", "slices")] \
            + [("pairs", ctypes.c_bool)]

    class Pack(ctypes.Structure):   # PackArgs of csrc/pack_weights.h
        _fields_ = [("p", ctypes.c_void_p * 8)] + [(n, ctypes.c_int) for n in ("D", "G", "Gp", "n_up", "n_out", "n_dw")]

    L = _lib.lib()
    plan = L["_ZN3pdw21dense_wide_first_planEPNS_9ColsumJobExiiiii"]
    plan.restype = ctypes.c_bool
    launch = L["_ZN3pdw23dense_wide_first_launchEPKvS1_PvS2_ixiiRKNS_9ColsumJobEPKNS_8PackArgsEiP12ihipStream_t"]
    (B, H, W, D), NO, k = shape, 2 * padded, 3
    N, dt = B * H * W, _lib.dtype_code(dtype)
    gen = torch.Generator(device="cuda").manual_seed(D)
    r = lambda *s: torch.randn(*s, generator=gen, device="cuda").to(dtype)
    x, w = r(*shape), (r(2 * half, D) / 16).to(dtype)
    given = [w, r(D, 2 * half), r(k, k, 2 * half), r(k, k, 2 * half)]
    wide = [torch.zeros(NO, D, device="cuda", dtype=dtype), *[torch.zeros(*s, NO, device="cuda", dtype=dtype) for s in ((D,), (k, k), (k, k))]]
    for i in range(2):
        a, b = slice(i * half, (i + 1) * half), slice(i * padded, i * padded + half)
        wide[0][b] = given[0][a]
        for q, t in zip(wide[1:], given[1:]):
            q[..., b] = t[..., a]
    packed = [torch.full_like(t, float("nan")) for t in wide]
    y, pool = torch.full((B, H, W, NO), float("nan"), device="cuda", dtype=dtype), torch.full((B, H // 2, W // 2, NO), float("nan"), device="cuda", dtype=dtype)
    at, sums = lambda t: ctypes.c_void_p(t.data_ptr()), Sums()
    assert plan(ctypes.byref(sums), ctypes.c_longlong(N), D, NO, B, H * W, dt)
    part = torch.full((B, sums.n, D), float("nan"), device="cuda")
    sums.x, sums.part = x.data_ptr(), part.data_ptr()
    pack = Pack((ctypes.c_void_p * 8)(*[t.data_ptr() for t in given + packed]), D, half, padded, NO * D // 8, NO * D // 8, k * k * NO // 8)
    assert launch(at(x), at(w), at(y), at(pool), W // 2, ctypes.c_longlong(N), D, NO, ctypes.byref(sums), ctypes.byref(pack) if half != padded else None, dt,
                  ctypes.c_void_p(_lib.stream_ptr(x.device))) == 0
    assert_close(y, (x.double().cpu().reshape(N, D) @ wide[0].double().cpu().t()).reshape(y.shape).numpy(), dtype, "y")
    q = y.float().reshape(B, H // 2, 2, W // 2, 2, NO)
    assert torch.equal(pool, ((((q[:, :, 0, :, 0] + q[:, :, 0, :, 1]) + q[:, :, 1, :, 0]) + q[:, :, 1, :, 1]) * 0.25).to(dtype))
    assert_close(part.double().sum(1).float(), x.double().sum((1, 2)).cpu().numpy(), torch.float32, "sums")
    if half != padded:
        assert all(torch.equal(a, b) for a, b in zip(packed, wide))
