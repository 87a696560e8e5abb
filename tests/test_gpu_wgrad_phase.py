"""The 16-bit weight gradient of the depthwise convolution against the float64 oracle at the edges of its kernels' tiles, its
partial sums inside the workspace that the size query names."""
import pytest
import torch

from parity import TOL, randn, rel_err

pytestmark = pytest.mark.gpu


def _wgrad(x, gy, k, pad, guard=1 << 20):
    """pdw_dwconv_wgrad through the C ABI into a workspace of exactly the size asked for, a guard area behind it."""
    from pyramidconvblock_amd import _lib

    L = _lib.lib()
    (B, H, W, C), code = x.shape, _lib.dtype_code(x.dtype)
    geo = (B, H, W, C, k, k, 1, 1, *pad, 1, 1)
    need = L.pdw_dwconv_wgrad_workspace_bytes(*geo, code)
    ws = torch.full((need // 4 + guard,), 7.0, device="cuda")
    dw = torch.full((k, k, C), float("nan"), device="cuda", dtype=x.dtype)
    _lib.check(L.pdw_dwconv_wgrad(x.data_ptr(), gy.data_ptr(), dw.data_ptr(), ws.data_ptr(), need, *geo, code,
                                  _lib.stream_ptr(x.device)), "pdw_dwconv_wgrad")
    torch.cuda.synchronize()
    assert bool((ws[need // 4:] == 7.0).all()), "partial sums beyond the workspace"
    return dw


def _check(oracle, shape, k, pad, dtype, seed):
    B, H, W, C = shape
    gen = torch.Generator().manual_seed(seed)
    x = randn(gen, *shape).to(dtype)
    gy = randn(gen, B, H + 2 * pad[0] - k + 1, W + 2 * pad[1] - k + 1, C).to(dtype)
    want = oracle.dwconv_wgrad(x.double().numpy(), gy.double().numpy(), (k, k), 1, pad, 1)
    assert rel_err(_wgrad(x.cuda(), gy.cuda(), k, pad), want) <= TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape,k", [((2, 40, 44, 64), 4), ((3, 17, 70, 24), 8), ((1, 20, 20, 16), 2), ((2, 24, 28, 8), 14),
                                     ((2, 24, 28, 16), 16)])
def test_even_filters(oracle, shape, k, dtype):
    _check(oracle, shape, k, (k // 2, k // 2), dtype, 10 * k)


# one tile column of 64, two, and columns of 32 in two images (an odd number of them); rows off and on multiples of the passes
# of 8; channels off the slices of 16; runs of rows that start and end inside an image; images smaller than the filter
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape,k", [((1, 8, 64, 16), 3), ((2, 9, 65, 24), 9), ((3, 57, 61, 8), 13), ((5, 16, 32, 40), 15),
                                     ((3, 7, 7, 16), 11), ((4, 33, 31, 16), 5), ((2, 15, 112, 24), 7), ((7, 24, 63, 16), 13),
                                     ((1, 1, 1, 8), 15), ((9, 3, 33, 8), 1), ((40, 28, 28, 32), 13), ((2, 70, 20, 136), 9),
                                     # one column and row more than an operand's 16
                                     ((1, 8, 64, 16), 17), ((3, 57, 61, 8), 17), ((5, 16, 32, 40), 17), ((1, 1, 1, 8), 17),
                                     ((40, 28, 28, 32), 17), ((2, 15, 112, 24), 17), ((3, 7, 7, 16), 17), ((2, 70, 20, 136), 17)])
def test_tiles_and_runs(oracle, shape, k, dtype):
    _check(oracle, shape, k, (k // 2, k // 2), dtype, k + shape[1])


@pytest.mark.parametrize("shape,k,pad", [((3, 20, 40, 16), 13, (0, 0)), ((2, 18, 34, 24), 9, (8, 8)), ((2, 17, 33, 8), 5, (7, 6)),
                                         ((3, 16, 70, 16), 15, (14, 3)), ((2, 13, 13, 16), 11, (1, 10)),
                                         ((2, 18, 34, 16), 17, (16, 0)), ((3, 20, 40, 16), 17, (3, 16)), ((2, 17, 70, 24), 16, (0, 15))])
def test_paddings_other_than_same(oracle, shape, k, pad):
    _check(oracle, shape, k, pad, torch.bfloat16, k + pad[0])
