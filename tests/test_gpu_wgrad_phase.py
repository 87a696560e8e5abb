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
