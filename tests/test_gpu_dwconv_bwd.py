"""Both gradients of a stand-alone depthwise convolution as one call (csrc/dwconv_bwd3.h without a pooled scale): against the float64
oracle and the two separate calls, with the partial sums inside the workspace that the size query names."""
import ctypes

import pytest
import torch

from parity import TOL, randn, rel_err

pytestmark = pytest.mark.gpu

# two results of one sum, each rounded to 16 bits once, are at most one unit in the last place apart (2^-7 and 2^-10 of the value at
# most), and near zero by what the order of fp32 additions makes of the largest terms
ULP = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 0.0}


def _both(x, gy, w, geo, guard=1 << 18):
    """(dx, dw) of pdw_dwconv_bwd and of the two calls."""
    from pyramidconvblock_amd import _lib

    L, code, s = _lib.lib(), _lib.dtype_code(x.dtype), _lib.stream_ptr(x.device)
    need = L.pdw_dwconv_wgrad_workspace_bytes(*geo, code)
    ws = torch.full((need // 4 + guard,), 7.0, device="cuda")
    dx, dw, dx2, dw2 = (torch.full_like(t, float("nan")) for t in (x, w, x, w))
    _lib.check(L.pdw_dwconv_bwd(gy.data_ptr(), w.data_ptr(), x.data_ptr(), dx.data_ptr(), dw.data_ptr(), ws.data_ptr(), need, *geo, code, s),
               "pdw_dwconv_bwd")
    torch.cuda.synchronize()
    assert bool((ws[need // 4:] == 7.0).all()), "partial sums beyond the workspace"
    _lib.check(L.pdw_dwconv_dgrad(gy.data_ptr(), w.data_ptr(), dx2.data_ptr(), *geo, code, s), "pdw_dwconv_dgrad")
    _lib.check(L.pdw_dwconv_wgrad(x.data_ptr(), gy.data_ptr(), dw2.data_ptr(), ws.data_ptr(), need, *geo, code, s), "pdw_dwconv_wgrad")
    return dx, dw, dx2, dw2


def _same(dx, dw, dx2, dw2):
    assert torch.equal(dx, dx2)
    a, b = dw.double(), dw2.double()
    assert bool(((a - b).abs() <= ULP[dw.dtype] * b.abs() + 1e-5 * b.abs().max()).all())


# one workgroup a problem; tiles of one image and of two (an odd number of them); channels off the slices; images smaller than the filter
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape,k", [((1, 1, 1, 8), 3), ((1, 8, 64, 16), 17), ((3, 7, 7, 24), 15), ((2, 33, 31, 40), 5), ((3, 57, 61, 8), 9),
                                     ((5, 16, 32, 40), 13), ((2, 15, 112, 24), 7), ((1, 20, 20, 16), 11)])
def test_against_the_oracle(oracle, shape, k, dtype):
    B, H, W, C = shape
    gen = torch.Generator().manual_seed(k + H)
    x, gy, w = randn(gen, *shape).to(dtype), randn(gen, *shape).to(dtype), randn(gen, k, k, C).to(dtype)
    p = (k // 2, k // 2)
    dx, dw, dx2, dw2 = _both(x.cuda(), gy.cuda(), w.cuda(), (B, H, W, C, k, k, 1, 1, *p, 1, 1))
    assert rel_err(dw, oracle.dwconv_wgrad(x.double().numpy(), gy.double().numpy(), (k, k), 1, p, 1)) <= TOL[dtype]
    _same(dx, dw, dx2, dw2)


# one round of workgroups, several rounds (72, 47 and 53 slices), runs across images and inside one, and sizes that keep two launches
@pytest.mark.parametrize("shape,k", [((8, 64, 64, 1152), 9), ((5, 92, 92, 752), 3), ((24, 34, 35, 848), 17), ((32, 28, 28, 256), 13),
                                     ((40, 7, 7, 264), 15), ((64, 56, 56, 128), 13), ((3, 62, 66, 360), 5), ((78, 11, 8, 1144), 7)])
def test_cuts(shape, k):
    gen = torch.Generator(device="cuda").manual_seed(k)
    x, gy = (torch.randn(shape, generator=gen, device="cuda").bfloat16() for _ in range(2))
    w = torch.randn(k, k, shape[3], generator=gen, device="cuda").bfloat16()
    _same(*_both(x, gy, w, (*shape, k, k, 1, 1, k // 2, k // 2, 1, 1)))


def _launches(x, gy, w, geo):
    """Kernels that a call of pdw_dwconv_bwd launches: the nodes of a graph that it is captured into (and that is not replayed)."""
    from pyramidconvblock_amd import _lib

    L, code = _lib.lib(), _lib.dtype_code(x.dtype)
    need = L.pdw_dwconv_wgrad_workspace_bytes(*geo, code)
    ws, dx, dw = torch.empty(need // 4 + 1, device="cuda"), torch.empty_like(x), torch.empty_like(w)
    stream = torch.cuda.Stream()

    def call():
        _lib.check(L.pdw_dwconv_bwd(gy.data_ptr(), w.data_ptr(), x.data_ptr(), dx.data_ptr(), dw.data_ptr(), ws.data_ptr(), need, *geo, code,
                                    stream.cuda_stream), "pdw_dwconv_bwd")

    torch.cuda.synchronize()
    call()
    torch.cuda.synchronize()
    hip = ctypes.CDLL("libamdhip64.so")
    handle, graph, nodes = ctypes.c_void_p(stream.cuda_stream), ctypes.c_void_p(), ctypes.c_size_t()
    assert hip.hipStreamBeginCapture(handle, 1) == 0   # (calls of this thread)
    try:
        call()
    finally:
        ended = hip.hipStreamEndCapture(handle, ctypes.byref(graph))
    assert ended == 0 and hip.hipGraphGetNodes(graph, None, ctypes.byref(nodes)) == 0
    assert hip.hipGraphDestroy(graph) == 0
    return nodes.value


# the shared launch and its summation, in one round of workgroups and in several (72, 69 and 66 slices); two launches and the summation where the
# shared one takes as long or longer: runs of the weight gradient twice as long to make room (45 slices), chips full of either
# side, one round estimated less than 6 % ahead (filter 7), or with runs of the weight gradient three times as long (filter 5)
@pytest.mark.parametrize("shape,k,launches", [((2, 20, 20, 64), 7, 2), ((32, 28, 28, 256), 13, 2), ((8, 64, 64, 1152), 9, 2), ((8, 19, 19, 1096), 7, 2),
                                              ((10, 16, 16, 1056), 9, 2), ((74, 17, 17, 896), 9, 3), ((40, 15, 15, 712), 13, 3),
                                              ((64, 56, 56, 128), 13, 3), ((39, 45, 45, 216), 17, 3),
                                              ((11, 64, 64, 432), 7, 3), ((92, 7, 7, 448), 5, 3)])
def test_launches(shape, k, launches):
    x, w = torch.zeros(shape, device="cuda", dtype=torch.bfloat16), torch.zeros(k, k, shape[3], device="cuda", dtype=torch.bfloat16)
    n = _launches(x, torch.zeros_like(x), w, (*shape, k, k, 1, 1, k // 2, k // 2, 1, 1))
    assert n == launches


# what the shared launch does not take runs as the two calls
@pytest.mark.parametrize("dtype,k,stride,pad,dil", [(torch.float32, 5, 1, 2, 1), (torch.bfloat16, 5, 2, 2, 1), (torch.bfloat16, 4, 1, 2, 1),
                                                    (torch.bfloat16, 5, 1, 0, 1), (torch.float16, 3, 1, 2, 2), (torch.bfloat16, 19, 1, 9, 1)])
def test_other_calls(dtype, k, stride, pad, dil):
    B, H, W, C = 2, 21, 24, 16
    oh, ow = ((n + 2 * pad - dil * (k - 1) - 1) // stride + 1 for n in (H, W))
    gen = torch.Generator(device="cuda").manual_seed(k)
    x, gy, w = (torch.randn(s, generator=gen, device="cuda").to(dtype) for s in ((B, H, W, C), (B, oh, ow, C), (k, k, C)))
    dx, dw, dx2, dw2 = _both(x, gy, w, (B, H, W, C, k, k, stride, stride, pad, pad, dil, dil))
    assert torch.equal(dx, dx2) and torch.equal(dw, dw2)


def test_module_graph_and_eager_agree():
    """A training step of the module as a graph, replayed between eager steps."""
    import pyramidconvblock_amd as pcb
    from pyramidconvblock_amd.graphs import GraphedStep

    torch.manual_seed(0)
    m = pcb.OptimizedDepthwiseConv2d(64, 7, padding=3).bfloat16().cuda()
    x, g = torch.randn(3, 20, 24, 64, device="cuda").bfloat16(), torch.randn(3, 20, 24, 64, device="cuda").bfloat16()
    step = GraphedStep(m, x, g)
    for i in range(3):
        step.replay()
        got = [step.x.grad.clone(), *[p.clone() for p in step.param_grads]]
        xe = x.clone().requires_grad_()
        want = torch.autograd.grad(m(xe), [xe, *m.parameters()], g)
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
