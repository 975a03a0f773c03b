"""The weight gradient of tall_matmul for gradients that are not plain matrices in
memory (batched by vmap, forward-mode duals, lazily negated views, a vector of
weights): they take the products of torch, on every device."""
import pytest
import torch
from torch.autograd import forward_ad
from torch.utils.flop_counter import FlopCounterMode

from stile_amd import autograd
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


def _batched(dev):
    H, W, dY = _operands(dev)
    dW, = torch.autograd.grad(tall_matmul(H, W), W, dY, is_grads_batched=True)
    assert dW.shape == (4, F, FG)
    for i in range(4):
        _check(H, dY[i], dW[i])


def _vmap(dev):
    H, W, dY = _operands(dev)
    y = tall_matmul(H, W)
    dW = torch.vmap(lambda d: torch.autograd.grad(y, W, d, retain_graph=True)[0])(dY)
    for i in range(4):
        _check(H, dY[i], dW[i])


def _dual(dev):
    H, W, dY = _operands(dev)
    y = tall_matmul(H, W)
    with forward_ad.dual_level():
        dW, = torch.autograd.grad(y, W, forward_ad.make_dual(dY[0], dY[1]))
        got = forward_ad.unpack_dual(dW)
        _check(H, dY[0], got.primal)
        assert got.tangent is not None
        _check(H, dY[1], got.tangent)


def _negated(dev):
    H, W, dY = _operands(dev)
    d = torch.complex(dY[0], dY[1]).conj().imag
    assert d.is_neg()
    dW, = torch.autograd.grad(tall_matmul(H, W), W, d)
    _check(H, -dY[1], dW)


def _vector(dev):
    H, _, dY = _operands(dev)
    w = torch.randn(F, device=dev, requires_grad=True)
    dw, = torch.autograd.grad(tall_matmul(H, w), w, dY[0, :, 0])
    assert dw.shape == (F,)
    _check(H, dY[0, :, :1], dw[:, None])


def _counted(dev):
    H, W, dY = _operands(dev)
    with FlopCounterMode(display=False) as mode:
        dW, = torch.autograd.grad(tall_matmul(H, W), W, dY[0])
    assert mode.get_total_flops() == 2 * (2 * M * F * FG)
    _check(H, dY[0], dW)


ROUTES = [_batched, _vmap, _dual, _negated, _vector, _counted]


@pytest.mark.parametrize("route", ROUTES)
def test_on_the_cpu(route):
    route("cpu")


@pytest.mark.gpu
@pytest.mark.parametrize("route", ROUTES)
def test_on_the_gpu(cuda, route):
    print("tall route", route.__name__, flush=True)
    route(cuda)


@pytest.mark.parametrize("route", [_batched, _vmap, _dual, _negated])
def test_operands_without_memory_of_their_own_are_told_apart(monkeypatch, route):
    seen = []

    def spy(H, G):
        seen.append(autograd._own_memory(G))
        return H.t() @ G

    monkeypatch.setattr(autograd, "_split_k_tn", spy)
    route("cpu")
    assert seen and not any(seen)
    H, W, dY = _operands("cpu")
    torch.autograd.grad(tall_matmul(H, W), W, dY[0])
    assert seen[-1]


@pytest.mark.gpu
def test_wide_products_are_the_gemms(cuda):
    """1024 x 1024 entries and 2048 x 512, which the GEMM has tiles enough for."""
    with torch.no_grad():
        H, G = torch.zeros(65552, 2048, device=cuda), torch.zeros(65552, 1024, device=cuda)
        assert not autograd._tall_kernel_fits(H[:, :1024], G)
        assert not autograd._tall_kernel_fits(H, G[:, :512])
        assert autograd._tall_kernel_fits(H[:, :768], G[:, :768])
