"""The non-finite contract of the depthwise convolution (include/pdw.h, "Non-finite inputs").

The reference masks its loads (dwconv_triton.py:55-86): an Inf or NaN pixel reaches exactly the K x K footprint of
the filter around it.  The kernels here multiply a window somewhat larger than the filter by zero-padded filter
operands, so the value may also turn nearby outputs into NaN (0 * Inf), by at most PDW_NONFINITE_REACH pixels in
every direction (the fp32 kernels: 5 on the matrix cores, 1 on the vector ALU).  These tests pin that: every output further away, and every other channel, must equal the
float64 oracle of the clean input to the usual tolerance; every output the reference makes non-finite must be
non-finite here as well.
"""
import re
from pathlib import Path

import numpy as np
import pytest
import torch

from parity import TOL, randn

pytestmark = pytest.mark.gpu

REACH = int(re.search(r"#define\s+PDW_NONFINITE_REACH\s+(\d+)", (Path(__file__).resolve().parents[1] / "include" / "pdw.h").read_text()).group(1))


def _box(shape_hw, pix, k, pad, reach):
    """Mask [H, W] of the outputs a value at input pixel `pix` reaches through a k x k 'same' filter, dilated."""
    H, W = shape_hw
    m = np.zeros((H, W), dtype=bool)
    i, j = pix
    # output (oi, oj) reads input (oi - pad + u, oj - pad + v), 0 <= u, v < k
    lo_i, hi_i = i + pad - (k - 1) - reach, i + pad + reach
    lo_j, hi_j = j + pad - (k - 1) - reach, j + pad + reach
    m[max(lo_i, 0):max(min(hi_i, H - 1) + 1, 0), max(lo_j, 0):max(min(hi_j, W - 1) + 1, 0)] = True
    return m


F32_REACH, F32_VECTOR_REACH = 5, 1   # of the fp32 kernels: on the matrix cores, on the vector ALU (within REACH, both)

CASES = [
    # shape, k, dtype, reach
    ((2, 40, 44, 64), 13, torch.bfloat16, REACH),   # matrix-core kernels, 16 patches per image row
    ((2, 40, 44, 64), 7, torch.float16, REACH),
    ((4, 28, 28, 64), 13, torch.bfloat16, REACH),   # two images side by side in one instruction
    ((2, 57, 61, 24), 9, torch.bfloat16, REACH),
    ((2, 30, 33, 100), 9, torch.bfloat16, REACH),   # C % 8 != 0: vector kernel, 16-bit dot products
    ((2, 30, 33, 20), 13, torch.float32, F32_REACH),    # fp32 matrix-core kernel: every filter from 13 on
    ((2, 40, 44, 8), 17, torch.float32, F32_REACH),
    ((2, 30, 33, 20), 7, torch.float32, F32_REACH),     # ... small tensors at the small filters
    ((2, 50, 52, 12), 11, torch.float32, F32_REACH),    # ... 9 and 11 on filled tiles
    ((5, 24, 16, 8), 15, torch.float32, F32_REACH),     # ... four images side by side, the last tile not full
    ((2, 60, 58, 60), 7, torch.float32, F32_VECTOR_REACH),    # fp32 vector kernel: a large tensor at a small filter,
    ((1, 90, 70, 60), 3, torch.float32, F32_VECTOR_REACH),
    ((2, 30, 33, 18), 13, torch.float32, F32_VECTOR_REACH),   # channels off multiples of 4,
    ((3, 24, 33, 20), 9, torch.float32, F32_VECTOR_REACH),    # images that leave half of a tile empty
    ((1, 24, 25, 16), 17, torch.float16, REACH),
]
PLANTS = [(0, 17, 19, 5, float("inf")), (1, 2, 1, 3, float("nan")), (0, 23, 0, 7, float("-inf"))]


@pytest.mark.parametrize("shape,k,dtype,reach", CASES)
def test_forward_and_input_gradient_footprint(oracle, shape, k, dtype, reach):
    from pyramidconvblock_amd.dwconv import dwconv_dgrad, dwconv_forward

    B, H, W, C = shape
    pad = k // 2
    gen = torch.Generator().manual_seed(k + C)
    x = randn(gen, B, H, W, C).to(dtype)
    w = (randn(gen, k, k, C) / k).to(dtype)
    geo = ((1, 1), (pad, pad), (1, 1))
    clean_fwd = oracle.dwconv_fwd(x.double().numpy(), w.double().numpy(), 1, (pad, pad), 1)
    clean_dg = oracle.dwconv_dgrad(x.double().numpy(), w.double().numpy(), (H, W), 1, (pad, pad), 1)
    xp = x.clone()
    plants = [p for p in PLANTS if p[0] < B and p[1] < H and p[2] < W and p[3] < C]
    for (b, i, j, c, v) in plants:
        xp[b, i, j, c] = v
    bad_fwd = oracle.dwconv_fwd(xp.double().numpy(), w.double().numpy(), 1, (pad, pad), 1)
    bad_dg = oracle.dwconv_dgrad(xp.double().numpy(), w.double().numpy(), (H, W), 1, (pad, pad), 1)
    for name, got, clean, bad, flip in (
        ("forward", dwconv_forward(xp.cuda(), w.cuda(), *geo), clean_fwd, bad_fwd, False),
        ("input gradient", dwconv_dgrad(xp.cuda(), w.cuda(), (B, H, W, C), *geo), clean_dg, bad_dg, True),
    ):
        got = got.float().cpu().numpy().astype(np.float64)
        may = np.zeros((B, H, W, C), dtype=bool)
        for (b, i, j, c, _) in plants:
            # forward: output o reads input o - pad + u; the input gradient is the same with the filter rotated
            # (pad' = k - 1 - pad = pad for odd k), so the box is the same
            may[b, :, :, c] |= _box((H, W), (i, j), k, pad, reach)
        # 1. away from the planted values: finite and equal to the clean oracle
        far = ~may
        assert np.isfinite(got[far]).all(), f"{name}: non-finite output beyond the stated reach"
        scale = np.abs(clean).max()
        err = np.abs(got[far] - clean[far]).max() / scale
        assert err <= TOL[dtype], f"{name}: outputs outside the reach differ from the clean oracle: {err}"
        # 2. where the reference's masked loads give a non-finite result, so does the kernel
        ref_bad = ~np.isfinite(bad)
        assert ref_bad.any()
        assert (~np.isfinite(got[ref_bad])).all(), f"{name}: a non-finite reference output came out finite"
        assert not (ref_bad & far).any()


@pytest.mark.parametrize("shape,k,dtype", [c[:3] for c in CASES[:5]] + [
    ((2, 30, 33, 20), 13, torch.float32), ((3, 24, 40, 12), 7, torch.float32), ((5, 16, 8, 16), 15, torch.float32),   # matrix cores
    ((4, 13, 11, 20), 9, torch.float32),   # vector ALU
])
def test_weight_gradient_other_channels_unaffected(oracle, shape, k, dtype):
    """A non-finite value in x or gy may make any tap of ITS channel non-finite (the reference: the taps whose shifted
    position falls inside the image, which is nearly all of them); the other channels must be untouched."""
    from pyramidconvblock_amd.dwconv import dwconv_wgrad

    B, H, W, C = shape
    pad = k // 2
    gen = torch.Generator().manual_seed(3 * k + C)
    x = randn(gen, B, H, W, C).to(dtype)
    g = randn(gen, B, H, W, C).to(dtype)
    geo = ((1, 1), (pad, pad), (1, 1))
    clean = oracle.dwconv_wgrad(x.double().numpy(), g.double().numpy(), (k, k), 1, (pad, pad), 1)
    xp, gp = x.clone(), g.clone()
    xp[0, 5, 6, 5] = float("inf")
    gp[B - 1, 3, 2, 9] = float("nan")
    bad = oracle.dwconv_wgrad(xp.double().numpy(), gp.double().numpy(), (k, k), 1, (pad, pad), 1)
    got = dwconv_wgrad(xp.cuda(), gp.cuda(), (k, k, C), *geo).float().cpu().numpy().astype(np.float64)
    others = np.ones(C, dtype=bool)
    others[[5, 9]] = False
    assert np.isfinite(got[:, :, others]).all()
    err = np.abs(got[:, :, others] - clean[:, :, others]).max() / np.abs(clean).max()
    assert err <= TOL[dtype], err
    ref_bad = ~np.isfinite(bad)
    assert ref_bad[:, :, [5, 9]].any() and not ref_bad[:, :, others].any()
    assert (~np.isfinite(got[ref_bad])).all()


# Images never meet: whatever one holds, the others' results are bitwise those of the clean batch.  (The 16-bit kernels walk a
# batch as one column of rows, and the last patch of an image multiplies up to three rows beyond its last window by zeros.)
HURT = 2   # an image with neighbours on both sides, in a batch side by side in pairs too
ODD = [3, 5, 7, 9, 11, 13, 15, 17]


def _hurt(t):
    t = t.clone()
    t[HURT] = float("nan")
    t[HURT, ..., ::2] = float("inf")
    return t


def _apart(what, got, want):
    others = [b for b in range(want.shape[0]) if b != HURT]
    assert torch.isfinite(want).all(), what
    assert torch.equal(got[others], want[others]), f"{what}: another image's values changed"


def _conv_results(x, w, pad):
    """Forward and input gradient, and both with the pool of the input or its gradient where the extents are even."""
    from pyramidconvblock_amd.dwconv import dwconv_dgrad, dwconv_forward

    geo = ((1, 1), (pad, pad), (1, 1))
    k, (B, H, W, C) = w.shape[0], x.shape
    res = {"forward": dwconv_forward(x, w, *geo)}
    if H + k - 1 - 2 * pad >= 1 and W + k - 1 - 2 * pad >= 1:   # (x as the gradient of a result)
        res["input gradient"] = dwconv_dgrad(x, w, (B, H + k - 1 - 2 * pad, W + k - 1 - 2 * pad, C), *geo)
    if 2 * pad == k - 1 and H % 2 == 0 and W % 2 == 0:
        res["forward of a pool"], res["pool"] = dwconv_forward(x, w, *geo, pool_to=(H // 2, W // 2))
        res["input gradient of a pool"] = dwconv_dgrad(x, w, (B, H, W, C), *geo, pooled_grad=x[:, ::2, ::2].contiguous())
    return res


@pytest.mark.parametrize("k", ODD)
@pytest.mark.parametrize("B,W,C,dtype", [(5, 20, 16, torch.bfloat16), (4, 44, 24, torch.float16), (4, 13, 20, torch.bfloat16),
                                         (5, 18, 12, torch.float32)])
def test_images_stay_apart(k, B, W, C, dtype):
    """Every height modulo 8, a run of rows to a part of an image; 20: two images side by side."""
    gen = torch.Generator().manual_seed(k + C)
    w = (randn(gen, k, k, C) / k).to(dtype).cuda()
    for H in [*range(1, 18), *range(22, 30)]:
        x = randn(gen, B, H, W, C).to(dtype).cuda()
        for pad in sorted({k // 2, 0, k - 1, k // 2 + 1}):
            if H + 2 * pad < k or W + 2 * pad < k:
                continue
            clean, hurt = _conv_results(x, w, pad), _conv_results(_hurt(x), w, pad)
            for name in clean:
                _apart(f"{name} k={k} H={H} pad={pad}", hurt[name], clean[name])


# heights after which a window row beyond the last one counts, by the filter, and one height of each filter where none does
LAST_ROWS = [(3, 5), (3, 6), (3, 7), (3, 14), (3, 8), (5, 13), (5, 14), (5, 12), (7, 13), (7, 16), (11, 9), (11, 10), (11, 11), (11, 28),
             (13, 9), (13, 58), (13, 40), (15, 57), (15, 17), (15, 20), (9, 14), (17, 14)]


@pytest.mark.parametrize("k,H", LAST_ROWS)
@pytest.mark.parametrize("B,W,C", [(40, 10, 136), (43, 36, 136), (4, 36, 16)])
def test_images_of_a_run_stay_apart(oracle, k, H, B, W, C):
    """The same where a run of rows crosses several images (more images x slices of channels than compute units), with the
    values of the other images against the clean oracle."""
    dtype, pad = torch.bfloat16, k // 2
    gen = torch.Generator().manual_seed(k + H)
    x, w = randn(gen, B, H, W, C).to(dtype), (randn(gen, k, k, C) / k).to(dtype)
    first, second = _conv_results(x.cuda(), w.cuda(), pad), _conv_results(_hurt(x).cuda(), w.cuda(), pad)
    for name in first:
        _apart(name, second[name], first[name])
    some = [b for b in (0, 1, 3, B - 1) if b < B]
    xs, ws = x[some].double().numpy(), w.double().numpy()
    for name, want in (("forward", oracle.dwconv_fwd(xs, ws, 1, (pad, pad), 1)),
                       ("input gradient", oracle.dwconv_dgrad(xs, ws, (H, W), 1, (pad, pad), 1))):
        got = second[name][some].double().cpu().numpy()
        assert np.abs(got - want).max() / np.abs(want).max() <= TOL[dtype], name


@pytest.mark.parametrize("shape,k", [((5, 14, 44, 64), 3), ((5, 28, 60, 64), 5), ((9, 13, 40, 64), 7), ((4, 18, 48, 128), 11), ((4, 58, 60, 128), 13),
                                     ((4, 57, 61, 64), 15), ((5, 34, 36, 64), 17), ((80, 14, 14, 256), 3), ((40, 7, 7, 520), 3)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_images_of_a_block_stay_apart(shape, k, dtype):
    """The shared launches of both scales, gates and mean branch, forward, backward and at inference."""
    import pyramidconvblock_amd as pcb

    torch.manual_seed(k)
    block = pcb.ConvBlock(dim=shape[3], kernel_size=k).to(dtype).cuda()
    gen = torch.Generator().manual_seed(k + shape[1])
    x, g = randn(gen, *shape).to(dtype).cuda(), randn(gen, *shape).to(dtype).cuda()

    def results(x, g):
        with torch.no_grad():
            inferred = block(x)
        x = x.clone().requires_grad_()
        y = block(x)
        torch.autograd.backward(y, g)
        return {"inference": inferred, "forward": y.detach(), "input gradient": x.grad}

    clean = results(x, g)
    for hurt in (results(_hurt(x), g), results(x, _hurt(g))):
        for name in clean:
            _apart(name, hurt[name], clean[name])
