"""The native host path of the operators (csrc/torch_ops.cpp) at the edges of what autograd may ask of it."""
import pytest
import torch

from parity import assert_close, randn
from test_gpu_block import _block_case
from test_gpu_modules import _block

pytestmark = pytest.mark.gpu


@pytest.fixture
def native_only(monkeypatch):
    """The block's Python form is out of reach."""
    from pyramidconvblock_amd import conv_block

    class Refuse:
        @staticmethod
        def apply(*a):
            raise AssertionError("the block went to its Python form")

    monkeypatch.setattr(conv_block, "ConvBlockFunction", Refuse)


@pytest.mark.parametrize("dim,k,shape", [(264, 5, (2, 9, 12, 264)), (512, 3, (3, 16, 16, 512)), (1032, 7, (1, 7, 9, 1032))])
def test_fp32_blocks_wider_than_256(oracle, native_only, dim, k, shape):
    _block_case(oracle, dim, k, shape, torch.float32)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("s", [2., 1.5, 0.75, 0.3])
@pytest.mark.parametrize("dim,shape", [(64, (2, 13, 18, 64)), (40, (3, 16, 34, 40)), (200, (1, 8, 9, 200))])
def test_second_scales_below_and_above_one(oracle, native_only, dtype, s, dim, shape):
    """Second scales that are not a half, enlarging ones among them (bins that overlap, a resize down)."""
    _block(oracle, dim, 7, shape, dtype, scales=(1., s))


@pytest.mark.parametrize("kind,dim,shape,dtype", [("block", 128, (2, 16, 32, 128), torch.bfloat16), ("block", 64, (2, 13, 18, 64), torch.float32),
                                                  ("conv", 64, (2, 13, 18, 64), torch.float16)])
def test_on_a_side_stream(kind, dim, shape, dtype):
    """Input and gradient written late on a side stream, the forward there, the backward asked for from the default stream:
    every kernel has to run on the forward's stream, behind what it reads."""
    import pyramidconvblock_amd

    torch.manual_seed(9)
    layer = (pyramidconvblock_amd.ConvBlock(dim=dim, kernel_size=5) if kind == "block"
             else pyramidconvblock_amd.OptimizedDepthwiseConv2d(dim, 5, padding=2)).to(dtype).cuda()
    x, g = (torch.randn(shape, device="cuda").to(dtype) for _ in range(2))
    x.requires_grad_()
    y = layer(x)
    want = [y, *torch.autograd.grad(y, [x, *layer.parameters()], g)]
    with torch.no_grad():
        plain = layer(x)
    late, late_g = torch.zeros_like(x, requires_grad=True), torch.zeros_like(g)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)
        with torch.no_grad():
            late.copy_(x)
            inferred = layer(late)
        y = layer(late)
        torch.cuda._sleep(20_000_000)
        late_g.copy_(g)
    torch.cuda.current_stream().wait_stream(side)
    got = [y, *torch.autograd.grad(y, [late, *layer.parameters()], late_g)]
    torch.cuda.synchronize()
    assert torch.equal(inferred, plain)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dim,k,shape,dtype", [
    (128, 13, (2, 24, 32, 128), torch.bfloat16),    # the fused launches
    (64, 7, (2, 13, 18, 64), torch.float32),        # the general sequence, pooled size not an exact half
    (200, 9, (1, 9, 7, 200), torch.float16),
])
def test_block_node_partial_gradients(oracle, dim, k, shape, dtype):
    """An input without gradient, frozen parameters, views as parameters and inputs, a second backward."""
    import pyramid_dwconv

    torch.manual_seed(7)
    m = pyramid_dwconv.ConvBlock(dim=dim, kernel_size=k).to(dtype)
    gen = torch.Generator().manual_seed(7)
    x, g = randn(gen, *shape).to(dtype), randn(gen, *shape).to(dtype)
    params = {n: p.detach().double().numpy() for n, p in m.state_dict().items()}
    yo, cache = oracle.convblock_fwd(x.double().numpy(), params)
    dxo, go = oracle.convblock_bwd(cache, g.double().numpy())
    m = m.cuda()
    m.conv_pool.weight.requires_grad_(False)
    base = torch.zeros(dim * dim + 1, dtype=dtype, device="cuda")      # conv_up's weight at an odd storage offset
    base[1:1 + m.conv_up.weight.numel()] = m.conv_up.weight.detach().flatten()
    m.conv_up.weight = torch.nn.Parameter(base[1:1 + m.conv_up.weight.numel()].view_as(m.conv_up.weight))
    xd = x.cuda().transpose(1, 2).contiguous().transpose(1, 2)           # not contiguous, no gradient
    y = m(xd)
    assert_close(y, yo, dtype, "y")
    torch.autograd.backward(y, g.cuda(), retain_graph=True)
    first = {n: p.grad.clone() for n, p in m.named_parameters() if p.grad is not None}
    assert set(first) == set(go) - {"conv_pool.weight"}
    for n, v in first.items():
        assert_close(v, go[n], dtype, "grad " + n)
    torch.autograd.backward(y, g.cuda())                                 # the kept graph once more: same bits, added
    for n, p in m.named_parameters():
        if p.grad is not None:
            assert torch.equal(p.grad, first[n] + first[n]), n
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.backward(y, g.cuda())
    xd = xd.requires_grad_()
    y = m(xd)
    torch.autograd.backward(y, g.cuda())
    assert_close(xd.grad, dxo, dtype, "dx")


def test_changed_in_place_is_noticed():
    import pyramid_dwconv
    import pyramidconvblock_amd

    m = pyramid_dwconv.ConvBlock(dim=64, kernel_size=5).bfloat16().cuda()
    conv = pyramidconvblock_amd.OptimizedDepthwiseConv2d(64, 5, padding=2).bfloat16().cuda()
    x = torch.randn(1, 8, 8, 64, device="cuda").bfloat16().requires_grad_()
    for layer, w in ((m, m.conv_up.weight), (conv, conv.weight)):
        y = layer(x)
        with torch.no_grad():
            w.add_(1)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            y.sum().backward()


@pytest.mark.parametrize("which", ["block", "conv"])
def test_a_copied_input_is_kept_as_copied(which):
    """An input that the kernels read from a dense copy: the backward uses that copy, whatever becomes of the input."""
    import pyramidconvblock_amd

    torch.manual_seed(5)
    layer = (pyramidconvblock_amd.ConvBlock(dim=64, kernel_size=5) if which == "block"
             else pyramidconvblock_amd.OptimizedDepthwiseConv2d(64, 5, padding=2)).float().cuda()
    flat = torch.randn(2 * 8 * 9 * 64 + 1, device="cuda")
    for x in (flat[:-1].view(2, 9, 8, 64).transpose(1, 2), flat[1:].view(2, 8, 9, 64)):   # strides, alignment
        leaves = [x.requires_grad_(), *layer.parameters()]
        y = layer(x)
        g = torch.randn_like(y)
        want = torch.autograd.grad(y, leaves, g, retain_graph=True)
        before = torch.cuda.memory_stats()["allocated_bytes.all.allocated"]
        got = torch.autograd.grad(y, leaves, g, retain_graph=True)
        again = torch.cuda.memory_stats()["allocated_bytes.all.allocated"] - before
        dense = x.detach().contiguous().clone().requires_grad_()
        yd = layer(dense)
        torch.autograd.grad(yd, [dense, *leaves[1:]], g, retain_graph=True)
        before = torch.cuda.memory_stats()["allocated_bytes.all.allocated"]
        torch.autograd.grad(yd, [dense, *leaves[1:]], g)
        assert again == torch.cuda.memory_stats()["allocated_bytes.all.allocated"] - before   # no second copy
        with torch.no_grad():
            flat.mul_(3)
        for a, b, c in zip(want, got, torch.autograd.grad(y, leaves, g)):
            assert torch.equal(a, b) and torch.equal(a, c)


class _NoGradient(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, g):
        return None


@pytest.mark.parametrize("kind,dim,shape,dtype", [("block", 128, (1, 8, 32, 128), torch.bfloat16), ("block", 64, (2, 7, 9, 64), torch.float32),
                                                  ("conv", 64, (2, 7, 9, 64), torch.float16)])
def test_no_gradient_from_behind_is_a_gradient_of_zero(kind, dim, shape, dtype):
    import pyramidconvblock_amd

    layer = (pyramidconvblock_amd.ConvBlock(dim=dim, kernel_size=5) if kind == "block"
             else pyramidconvblock_amd.OptimizedDepthwiseConv2d(dim, 5, padding=2)).to(dtype).cuda()
    x = torch.randn(shape, device="cuda").to(dtype).requires_grad_()
    _NoGradient.apply(layer(x)).sum().backward()
    for t in (x, *layer.parameters()):
        assert t.grad is not None and not t.grad.any()


@pytest.mark.parametrize("which", ["block", "conv"])
def test_a_hook_that_returns_another_tensor_is_refused(which):
    """The backward's kernels take addresses of what was saved: a saved-tensor hook that gives back something else (left on
    the host, cut short) ends in an error and not in a read out of bounds; one of another type is converted."""
    import pyramidconvblock_amd

    layer = (pyramidconvblock_amd.ConvBlock(dim=64, kernel_size=5) if which == "block"
             else pyramidconvblock_amd.OptimizedDepthwiseConv2d(64, 5, padding=2)).float().cuda()
    x = torch.randn(2, 7, 9, 64, device="cuda", requires_grad=True)
    for unpack in (lambda t: t.cpu(), lambda t: t[:-1], lambda t: t.flatten()[::2]):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
            y = layer(x)
        with pytest.raises(RuntimeError, match="came back as another one"):
            y.sum().backward()
    inputs = [x, *layer.parameters()]
    want = torch.autograd.grad(layer(x).sum(), inputs)
    with torch.autograd.graph.save_on_cpu():   # the hook in use: another tensor of the same kind
        y = layer(x)
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(y.sum(), inputs), want))
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.half(), lambda t: t):   # x and the weights in 16 bits
        y = layer(x)
    for a, b in zip(torch.autograd.grad(y.sum(), inputs), want):
        assert_close(a, b.double().cpu().numpy(), torch.float16, "gradient")


def _layers():
    import pyramid_dwconv
    import pyramidconvblock_amd

    torch.manual_seed(3)
    return [pyramid_dwconv.ConvBlock(dim=64, kernel_size=5).float().cuda(),
            pyramidconvblock_amd.OptimizedDepthwiseConv2d(64, 5, padding=2).float().cuda()]


@pytest.mark.parametrize("which", [0, 1])
def test_recomputed_under_a_checkpoint(which):
    """The unpacking of what the node saved runs the checkpointed forward again, recorded, layers of torch's own among it."""
    from torch.utils.checkpoint import checkpoint

    layer = _layers()[which]
    m = torch.nn.Sequential(torch.nn.Linear(64, 64), torch.nn.GELU(), layer).cuda()
    x = torch.randn(2, 8, 8, 64, device="cuda", requires_grad=True)
    inputs = [x, *m.parameters()]
    g = torch.randn(2, 8, 8, 64, device="cuda")
    plain = torch.autograd.grad(m(x), inputs, g)
    again = torch.autograd.grad(checkpoint(m, x, use_reentrant=False), inputs, g)
    for a, b in zip(plain, again):
        assert (a - b).abs().max() <= 1e-6 * a.abs().max()


@pytest.mark.parametrize("which", [0, 1])
def test_transforms_without_a_rule_are_refused(which):
    import torch.autograd.forward_ad as fwad

    layer = _layers()[which]
    x = torch.randn(2, 8, 8, 64, device="cuda")
    with fwad.dual_level(), pytest.raises(RuntimeError):
        layer(fwad.make_dual(x, torch.ones_like(x)))
    with pytest.raises(RuntimeError):
        torch.func.vmap(layer)(x[None])


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("kind,dim,k,shape,dtype", [
    ("block", 128, 13, (2, 24, 32, 128), torch.bfloat16),   # the fused launches, with an inference form
    ("block", 64, 7, (2, 13, 18, 64), torch.float32),       # the general sequence
    ("conv", 64, 5, (2, 9, 12, 64), torch.float16),
])
def test_a_trace_computes_again(kind, dim, k, shape, dtype, grad):
    """A module recorded by torch.jit.trace, on another input than the one it was traced with: the module's own result,
    and its gradients."""
    import pyramidconvblock_amd

    torch.manual_seed(3)
    layer = (pyramidconvblock_amd.ConvBlock(dim=dim, kernel_size=k) if kind == "block"
             else pyramidconvblock_amd.OptimizedDepthwiseConv2d(dim, k, padding=k // 2)).to(dtype).cuda()
    gen = torch.Generator().manual_seed(4)
    first, x, g = (randn(gen, *shape).to(dtype).cuda() for _ in range(3))
    x.requires_grad_(grad)
    with torch.set_grad_enabled(grad):
        traced = torch.jit.trace(layer, (first.requires_grad_(grad),), check_trace=False)
        want, got = layer(x), traced(x)
    assert_close(got, want.detach().double().cpu().numpy(), dtype, "y")
    if grad:
        inputs = [x, *layer.parameters()]
        for a, b in zip(torch.autograd.grad(got, inputs, g), torch.autograd.grad(want, inputs, g)):
            assert_close(a, b.double().cpu().numpy(), dtype, "gradient")
