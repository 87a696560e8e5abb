"""Both products that read a layer's output gradient as one launch, inside the block calls of widths that the tiled 16-bit layers
do not take."""
import pytest
import torch

from parity import TOL, randn, rel_err

pytestmark = pytest.mark.gpu


# (rows, M, NO): tiles of 64 rows and 128, 192 columns; fp32 up to 256 wide (no LDS), beyond, remainders of every tile, one row
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
