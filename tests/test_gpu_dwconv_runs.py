"""The 16-bit forward and input gradient where their runs of rows start and end: batches stacked into one column of rows, runs
that begin inside an image, cross several, or end between two; odd batches of narrow images (two side by side); paddings on
either side of a multiple of 8 rows."""
import pytest
import torch

from parity import TOL, randn, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,k,pad", [((40, 9, 40, 16), 5, 2), ((37, 7, 7, 136), 9, 4), ((300, 3, 20, 8), 3, 1),
                                         ((66, 20, 36, 64), 13, 6), ((5, 57, 61, 24), 17, 8), ((9, 16, 64, 272), 7, 3),
                                         ((3, 24, 112, 48), 15, 7), ((130, 8, 33, 8), 11, 5), ((6, 17, 30, 24), 9, 0),
                                         ((4, 12, 13, 40), 5, 11)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_runs_over_stacked_images(oracle, shape, k, pad, dtype):
    from pyramidconvblock_amd.dwconv import dwconv_dgrad, dwconv_forward

    B, H, W, C = shape
    gen = torch.Generator().manual_seed(k + H)
    x, w = randn(gen, *shape).to(dtype), (randn(gen, k, k, C) / k).to(dtype)
    gy = randn(gen, B, H + 2 * pad - k + 1, W + 2 * pad - k + 1, C).to(dtype)
    geo = ((1, 1), (pad, pad), (1, 1))
    want = oracle.dwconv_fwd(x.double().numpy(), w.double().numpy(), 1, (pad, pad), 1)
    assert rel_err(dwconv_forward(x.cuda(), w.cuda(), *geo), want) <= TOL[dtype]
    want = oracle.dwconv_dgrad(gy.double().numpy(), w.double().numpy(), (H, W), 1, (pad, pad), 1)
    assert rel_err(dwconv_dgrad(gy.cuda(), w.cuda(), shape, *geo), want) <= TOL[dtype]


@pytest.mark.parametrize("shape,k,pad", [((3, 30011, 9, 8), 5, 2), ((1, 40003, 33, 16), 3, 1), ((2, 65530, 7, 8), 9, 4), ((5, 29990, 11, 24), 7, 0)])
def test_tall_images_run_by_image(oracle, shape, k, pad):
    """Images too tall for a stack: runs are parts of an image of any length, the last one shorter."""
    from pyramidconvblock_amd.dwconv import dwconv_dgrad, dwconv_forward

    dtype = torch.bfloat16
    gen = torch.Generator().manual_seed(k)
    x, w = randn(gen, *shape).to(dtype), (randn(gen, k, k, shape[3]) / k).to(dtype)
    B, H, W, C = shape
    gy = randn(gen, B, H + 2 * pad - k + 1, W + 2 * pad - k + 1, C).to(dtype)
    geo = ((1, 1), (pad, pad), (1, 1))
    want = oracle.dwconv_fwd(x.double().numpy(), w.double().numpy(), 1, (pad, pad), 1)
    assert rel_err(dwconv_forward(x.cuda(), w.cuda(), *geo), want) <= TOL[dtype]
    want = oracle.dwconv_dgrad(gy.double().numpy(), w.double().numpy(), (H, W), 1, (pad, pad), 1)
    assert rel_err(dwconv_dgrad(gy.cuda(), w.cuda(), shape, *geo), want) <= TOL[dtype]


@pytest.mark.parametrize("shape", [(9, 2, 12, 32), (40, 2, 40, 64), (5, 3, 7, 48), (70, 3, 64, 32)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_images_shorter_than_a_step(oracle, shape, dtype):
    """Stacks with whole steps of 8 rows between images of two and three, where the runs' offsets pass the last image: the input
    gradient with a pooled one, and the gated convolutions of inference."""
    import pyramidconvblock_amd as pcb
    from pyramidconvblock_amd.dwconv import dwconv_dgrad

    B, H, W, C = shape
    gen = torch.Generator().manual_seed(H + W)
    for k in (15, 17):
        geo = ((1, 1), (k // 2, k // 2), (1, 1))
        if H % 2 == 0:
            gy, gp, w = randn(gen, *shape).to(dtype), randn(gen, B, H // 2, W // 2, C).to(dtype), (randn(gen, k, k, C) / k).to(dtype)
            want = oracle.dwconv_dgrad(gy.double().numpy(), w.double().numpy(), (H, W), 1, k // 2, 1)
            got = dwconv_dgrad(gy.cuda(), w.cuda(), shape, *geo, pooled_grad=gp.cuda())
            assert rel_err(got, want + oracle.avgpool_bwd(gp.double().numpy(), (H, W))) <= TOL[dtype]
        torch.manual_seed(k)
        m = pcb.ConvBlock(dim=C, kernel_size=k).to(dtype)
        x = randn(gen, *shape).to(dtype)
        params = {n: p.detach().double().numpy() for n, p in m.state_dict().items()}
        want, _ = oracle.convblock_fwd(x.double().numpy(), params)
        with torch.no_grad():
            assert rel_err(m.cuda()(x.cuda()), want) <= TOL[dtype]


@pytest.mark.parametrize("k", [3, 5, 15, 17])
@pytest.mark.parametrize("H,W,C", [(2, 12, 16), (6, 64, 24), (7, 40, 8), (8, 20, 48), (9, 9, 16), (16, 70, 40), (14, 14, 264)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_short_runs(k, H, W, C, dtype):
    """Few images, whose runs are one or two steps long, by themselves and in a batch of long runs: the same bits."""
    from pyramidconvblock_amd.dwconv import dwconv_dgrad, dwconv_forward

    B, few = 12000 * 64 // (H * W * C) * 16 + 40, 5
    gen = torch.Generator().manual_seed(k + H)
    w, geo = (randn(gen, k, k, C) / k).to(dtype).cuda(), ((1, 1), (k // 2, k // 2), (1, 1))
    gen = torch.Generator("cuda").manual_seed(k + H)
    x = torch.randn(B, H, W, C, generator=gen, device="cuda").to(dtype)
    assert torch.equal(dwconv_forward(x[:few], w, *geo), dwconv_forward(x, w, *geo)[:few])
    assert torch.equal(dwconv_dgrad(x[:few], w, x[:few].shape, *geo), dwconv_dgrad(x, w, x.shape, *geo)[:few])
    if H % 2 == 0 and W % 2 == 0:
        gp = torch.randn(B, H // 2, W // 2, C, generator=gen, device="cuda").to(dtype)
        whole = dwconv_dgrad(x, w, x.shape, *geo, pooled_grad=gp)
        assert torch.equal(dwconv_dgrad(x[:few], w, x[:few].shape, *geo, pooled_grad=gp[:few]), whole[:few])


@pytest.mark.parametrize("k", [3, 5, 15, 17])
@pytest.mark.parametrize("H,W,C", [(2, 12, 16), (7, 40, 48), (8, 20, 32), (13, 64, 16)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_short_gated_runs(k, H, W, C, dtype):
    """The same of the convolution with the gate in its store."""
    from pyramidconvblock_amd import _lib

    L = _lib.lib()
    B, few = 12000 * 64 // (H * W * C) * 16 + 40, 5
    gen = torch.Generator("cuda").manual_seed(k + H)
    x, w = torch.randn(B, H, W, C, generator=gen, device="cuda").to(dtype), (torch.randn(k, k, C, generator=gen, device="cuda") / k).to(dtype)

    def gated(x):
        y = torch.empty(*x.shape[:3], C // 2, device="cuda", dtype=dtype)
        _lib.check(L.pdw_dwconv_fwd_gate(x.data_ptr(), w.data_ptr(), y.data_ptr(), None, len(x), H, W, C, k, k // 2, 0, 0, _lib.dtype_code(dtype),
                                         _lib.stream_ptr(x.device)))
        return y

    assert torch.equal(gated(x[:few]), gated(x)[:few])


def test_plans_are_kept_by_shape():
    """More shapes than are kept, twice over and from two threads: every batch gives the results of the whole one."""
    from concurrent.futures import ThreadPoolExecutor

    from pyramidconvblock_amd.dwconv import dwconv_forward

    gen = torch.Generator().manual_seed(0)
    geo = ((1, 1), (1, 1), (1, 1))
    x, w = randn(gen, 300, 5, 7, 16).to(torch.bfloat16).cuda(), randn(gen, 3, 3, 16).to(torch.bfloat16).cuda()
    whole = dwconv_forward(x, w, geo[0], geo[1], geo[2])

    def batches(order):
        return all(torch.equal(dwconv_forward(x[:b], w, *geo), whole[:b]) for b in order for _ in range(2))

    with ThreadPoolExecutor(2) as pool:
        assert all(pool.map(batches, [range(1, 301), range(300, 0, -1)]))
