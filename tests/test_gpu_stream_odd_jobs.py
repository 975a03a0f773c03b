"""Streaming kernel with two windows side by side in a workgroup and an odd number
of (window, 64 columns): the last workgroup has one window for its eight waves."""
import pytest
import torch

from stile_amd import _native

from .test_gpu_stream_windows import _check, _operand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blocks,b", [("float32", "float32"), ("float16", "bfloat16"), ("bfloat16", "bfloat16")])
@pytest.mark.parametrize("sparse", [[0], [0, 3, 1], [2]])
@pytest.mark.parametrize("W,N,pad", [(601, 64, 0), (601, 63, 2), (513, 40, 0), (205, 192, 1)])
def test_last_workgroup_half_empty(cuda, blocks, b, sparse, W, N, pad):
    A, pack = _operand(1100, [20, 40, 33] * (W // 3) + [5] * (W % 3), sparse, W)
    assert W * -(-N // 64) >= 512 and W * -(-N // 64) % 2 == 1
    plan = _native.Plan.spmm(pack, blocks)
    g = torch.Generator(device=cuda)
    g.manual_seed(N)
    B = torch.randn(1100, N + pad, device=cuda, generator=g).to(getattr(torch, b))[:, :N]
    out = torch.full((16 * W, N + 5), 7.0, device=cuda)
    print("stream odd jobs", blocks, b, sparse, W, N, pad, flush=True)
    _check(A, B, plan.run_spmm(B, out[:, :N]), blocks)
    assert torch.all(out[:, N:] == 7.0)
