"""Both products that read a layer's output gradient as one launch, inside the block calls of widths that the tiled 16-bit layers
do not take."""
import ctypes

import pytest
import torch

from parity import TOL, assert_close, randn, rel_err

pytestmark = pytest.mark.gpu


# 16-bit tiles of 64 and 128 rows by 128 columns; fp32 up to 256 wide (no LDS) and beyond; remainders of every tile
@pytest.mark.parametrize("dtype,dim,shape", [(torch.bfloat16, 200, (3, 17, 19)), (torch.float16, 1152, (1, 16, 16)),
                                             (torch.bfloat16, 520, (2, 70, 66)), (torch.float32, 64, (2, 9, 7)),
                                             (torch.float32, 200, (1, 33, 20)), (torch.float32, 520, (1, 12, 13)),
                                             (torch.bfloat16, 136, (1, 4, 4)), (torch.float32, 24, (1, 4, 4))])
def test_block_gradients_through_the_pair(oracle, dtype, dim, shape):
    import pyramidconvblock_amd as pcb

    torch.manual_seed(dim)
    m = pcb.ConvBlock(dim=dim, kernel_size=3).to(dtype)
    gen = torch.Generator().manual_seed(7)
    x, g = (randn(gen, *shape, dim).to(dtype) for _ in range(2))
    params = {n: p.detach().double().numpy() for n, p in m.state_dict().items()}
    yo, cache = oracle.convblock_fwd(x.double().numpy(), params)
    dxo, go = oracle.convblock_bwd(cache, g.double().numpy())
    m = m.cuda()
    xd = x.cuda().requires_grad_()
    torch.autograd.backward(m(xd), g.cuda())
    assert rel_err(xd.grad, dxo) <= TOL[dtype]
    for n, p in m.named_parameters():
        assert rel_err(p.grad, go[n]) <= TOL[dtype], n


# 16-bit tiles of the input gradient 64 x 128, 128 x 128 and 128 x 192 beside 128 x 128 of the weight gradient; fp32 up to 256 wide
# and beyond; remainders of every tile, and one row
@pytest.mark.parametrize("dtype,N,M,NO", [(torch.bfloat16, 1, 136, 200), (torch.float16, 70, 264, 136), (torch.bfloat16, 33001, 136, 264),
                                          (torch.float16, 13185, 264, 576), (torch.bfloat16, 13185, 264, 576), (torch.float32, 1, 24, 32),
                                          (torch.float32, 129, 200, 104), (torch.float32, 1, 300, 260), (torch.float32, 1100, 520, 264)])
def test_the_shared_launch_itself(dtype, N, M, NO):
    """The launch behind the block calls (it has no C entry of its own): taken, and not left to two others, at every tile it has."""
    from pyramidconvblock_amd import _lib, ops

    lib = _lib.lib()
    launch = lib["_ZN3pdw21dense_bwd_both_launchEPKvS1_S1_PvS2_S2_mPKfixiiiP12ihipStream_t"]
    ptr, i64, i32 = ctypes.c_void_p, ctypes.c_longlong, ctypes.c_int
    launch.argtypes, launch.restype = [ptr] * 6 + [ctypes.c_size_t, ptr, i32, i64, i32, i32, i32, ptr], i32
    gen = torch.Generator().manual_seed(N + M)
    P = max(1, N // 3)
    g, x, w = randn(gen, N, M).to(dtype), randn(gen, N, NO).to(dtype), (randn(gen, M, NO) / M ** 0.5).to(dtype)
    rb = randn(gen, (N + P - 1) // P, NO)
    gd, xd, wd, rbd = g.cuda(), x.cuda(), w.cuda(), rb.cuda()
    dx, dw = torch.empty_like(xd), torch.empty_like(wd)
    ws = torch.empty(lib.pdw_dense_wgrad_workspace_bytes(N, M, NO), dtype=torch.uint8, device="cuda")
    with _lib.on_device(gd.device):
        status = launch(gd.data_ptr(), wd.data_ptr(), xd.data_ptr(), dx.data_ptr(), dw.data_ptr(), ws.data_ptr(), ws.numel(), rbd.data_ptr(), P, N,
                        M, NO, _lib.dtype_code(dtype), _lib.stream_ptr(gd.device))
    assert status == 0, status
    assert_close(dx, (g.double() @ w.double() + rb.double().repeat_interleave(P, 0)[:N]).numpy(), dtype, "input gradient", 0.5)
    assert_close(dw, (g.double().t() @ x.double()).numpy(), dtype, "weight gradient", 0.5)
    assert torch.equal(dw, ops.dense_wgrad(gd, xd))
