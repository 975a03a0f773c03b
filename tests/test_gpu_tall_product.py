"""H^T G of tall FP32 operands (the dense weight gradient) at the edges of its
128 x 64 tiles, row pairs and slabs, with strides and alignments that take either
load path, and through tall_matmul's backward.

Bound per element: (M + 2) 2^-24 sum|h||g| (M products, each rounded once and
added in FP32 in some order)."""
import pytest
import torch

from stile_amd import _native
from stile_amd.autograd import tall_matmul

pytestmark = pytest.mark.gpu


def _check(H, G, got):
    H64, G64 = H.double(), G.double()
    bound = (H.shape[0] + 2) * 2.0 ** -24 * (H64.abs().t() @ G64.abs())
    assert torch.all((got.double() - H64.t() @ G64).abs() <= bound)


@pytest.mark.parametrize("M", [1, 2, 3, 31, 127, 128, 129, 1000, 4097, 70001])
@pytest.mark.parametrize("F,Fg,pad", [(1, 1, 0), (3, 5, 2), (64, 64, 0), (128, 64, 0), (129, 65, 0), (132, 66, 4),
                                      (256, 200, 0), (40, 8, 1)])
def test_tile_and_slab_edges(cuda, M, F, Fg, pad):
    g = torch.Generator(device=cuda)
    g.manual_seed(M + F)
    H = torch.randn(M, F + pad, device=cuda, generator=g)[:, :F]
    G = torch.randn(M, Fg + pad, device=cuda, generator=g)[:, :Fg]
    print("tall", M, F, Fg, pad, flush=True)
    _check(H, G, _native.tall_tn_f32(H, G))


def test_backward_of_tall_matmul(cuda):
    H = torch.randn(9000, 48, device=cuda, requires_grad=True)
    W = torch.randn(48, 30, device=cuda, requires_grad=True)
    dY = torch.randn(9000, 30, device=cuda)
    print("tall backward", flush=True)
    dH, dW = torch.autograd.grad(tall_matmul(H, W), (H, W), dY)
    _check(H.detach(), dY, dW)
    # a gradient that is one value seen through strides of 0, and a transposed one
    dW, = torch.autograd.grad(tall_matmul(H, W).sum(), (W,))
    _check(H.detach(), torch.ones(9000, 30, device=cuda), dW)
    dT = torch.randn(30, 9000, device=cuda).t()
    dW, = torch.autograd.grad(tall_matmul(H, W), (W,), dT)
    _check(H.detach(), dT.contiguous(), dW)


def test_gradient_of_the_gradient(cuda):
    H = torch.randn(5000, 6, device=cuda, requires_grad=True)
    W = torch.randn(6, 4, device=cuda, requires_grad=True)
    dY = torch.randn(5000, 4, device=cuda, requires_grad=True)
    dW, = torch.autograd.grad(tall_matmul(H, W), (W,), dY, create_graph=True)
    dH, = torch.autograd.grad(dW.sum(), (H,))
    assert torch.allclose(dH, dY.detach().sum(1, keepdim=True).expand_as(dH), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("M", [65536, 131072, 131073, 262143, 262144])
@pytest.mark.parametrize("F,Fg", [(24, 32), (256, 256)])
def test_backward_where_row_slabs_take_over(cuda, M, F, Fg):
    g = torch.Generator(device=cuda)
    g.manual_seed(M + F)
    H = torch.randn(M, F, device=cuda, generator=g, requires_grad=True)
    W = torch.randn(F, Fg, device=cuda, generator=g, requires_grad=True)
    dY = torch.randn(M, Fg, device=cuda, generator=g)
    print("tall backward", M, F, Fg, flush=True)
    _check(H.detach(), dY, torch.autograd.grad(tall_matmul(H, W), W, dY)[0])
