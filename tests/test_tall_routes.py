"""The weight gradient of tall_matmul for gradients that are not plain matrices in
memory (batched by vmap, forward-mode duals, lazily negated views, a vector of
weights): they take the products of torch, on every device."""
import pytest
import torch

from stile_amd.autograd import tall_matmul

M, F, FG = 4100, 12, 9  # rows beyond those from which the library's kernel runs


def _operands(dev):
    g = torch.Generator().manual_seed(3)
    H = torch.randn(M, F, generator=g).to(dev)
    W = torch.randn(F, FG, generator=g).to(dev).requires_grad_(True)
    return H, W, torch.randn(4, M, FG, generator=g).to(dev)


def _check(H, G, got):
    """(M + 2) 2^-24 sum|h||g| per element: M products, each rounded once and
    added in FP32 in some order."""
    H64, G64 = H.cpu().double(), G.cpu().double()
    bound = (M + 2) * 2.0 ** -24 * (H64.abs().t() @ G64.abs())
    assert torch.all((got.detach().cpu().double() - H64.t() @ G64).abs() <= bound)


def _vector(dev):
    H, _, dY = _operands(dev)
    w = torch.randn(F, device=dev, requires_grad=True)
    dw, = torch.autograd.grad(tall_matmul(H, w), w, dY[0, :, 0])
    assert dw.shape == (F,)
    _check(H, dY[0, :, :1], dw[:, None])


ROUTES = [_vector]


@pytest.mark.parametrize("route", ROUTES)
def test_on_the_cpu(route):
    route("cpu")


@pytest.mark.gpu
@pytest.mark.parametrize("route", ROUTES)
def test_on_the_gpu(cuda, route):
    print("tall route", route.__name__, flush=True)
    route(cuda)
