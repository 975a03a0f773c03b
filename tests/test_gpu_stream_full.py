"""Full launches of the streaming kernels (a wave per window and 64 columns, a
workgroup per longer window): windows of up to two chunks in sequence at any size,
longer ones where there are enough of them, huge windows in parts beside them, few
sparse rows left to the row tasks, widths around 64 columns, unaligned rows and a B
that 24-bit row offsets cannot address.  Bounds as in test_gpu_stream_windows."""
import pytest
import torch

from stile_amd import _native

from .test_gpu_stream_windows import _check, _operand

pytestmark = pytest.mark.gpu

TYPES = [("float32", "float32"), ("float32", "bfloat16"), ("float16", "float16"), ("float16", "float32"),
         ("float16", "bfloat16"), ("bfloat16", "bfloat16"), ("bfloat16", "float32"), ("bfloat16", "float16")]


def _run(cuda, A, pack, blocks, b, N, pad=0):
    plan = _native.Plan.spmm(pack, blocks)
    g = torch.Generator(device=cuda)
    g.manual_seed(N)
    B = torch.randn(A.shape[1], N + pad, device=cuda, generator=g).to(getattr(torch, b))[:, :N]
    out = torch.full((A.shape[0], N + 5), 7.0, device=cuda)
    print("stream full", blocks, b, A.shape, N, pad, flush=True)
    _check(A, B, plan.run_spmm(B, out[:, :N]), blocks)
    assert torch.all(out[:, N:] == 7.0)
    once, again = plan.run_spmm(B, deterministic=True), plan.run_spmm(B, deterministic=True)
    _check(A, B, once, blocks)
    assert torch.equal(once, again)
    return plan


@pytest.mark.parametrize("blocks,b", TYPES)
@pytest.mark.parametrize("N,pad", [(1, 0), (63, 2), (64, 0), (65, 3), (132, 0), (321, 30)])
def test_two_chunks_in_sequence(cuda, blocks, b, N, pad):
    A, pack = _operand(1300, [1, 16, 32, 33, 64, 257, 288, 400, 512, 20, 5], [0], 1)
    _run(cuda, A, pack, blocks, b, N, pad)


@pytest.mark.parametrize("blocks,b", [("float32", "float32"), ("float16", "bfloat16"), ("bfloat16", "bfloat16")])
@pytest.mark.parametrize("N,pad", [(64, 0), (61, 1)])
def test_many_longer_windows(cuda, blocks, b, N, pad):
    A, pack = _operand(1100, [20, 100, 33, 250, 160] * 310 + [300, 600], [0], 2)
    _run(cuda, A, pack, blocks, b, N, pad)


@pytest.mark.parametrize("blocks,b", [("float32", "float32"), ("bfloat16", "bfloat16")])
@pytest.mark.parametrize("N,pad", [(96, 0), (99, 2)])
def test_parts_of_a_huge_window(cuda, blocks, b, N, pad):
    A, pack = _operand(9000, [8700, 300] + [20, 70, 100] * 270, [0], 3)
    _run(cuda, A, pack, blocks, b, N, pad)


@pytest.mark.parametrize("blocks,b", [("float32", "float32"), ("bfloat16", "bfloat16")])
def test_few_sparse_rows_beside(cuda, blocks, b):
    A, pack = _operand(1100, [20] * 2700, [5] + [0] * (16 * 2699) + [100] + [0] * 14, 4)
    assert _run(cuda, A, pack, blocks, b, 64).info()["sparse_nnz"] == 105


@pytest.mark.parametrize("blocks,b", [("float32", "float32"), ("bfloat16", "bfloat16")])
def test_rows_beyond_24_bit_offsets(cuda, blocks, b):
    ld = 1 << 23  # 2^24 bytes and more per row, 1100 rows: 18 / 35 GB
    A, pack = _operand(1100, [40, 300, 512], [0], 9)
    plan = _native.Plan.spmm(pack, blocks)
    B = torch.empty(1100, ld, device=cuda, dtype=getattr(torch, b))[:, :70]
    B.copy_(torch.randn(1100, 70, device=cuda))
    print("stream full wide rows", blocks, flush=True)
    _check(A, B, plan.run_spmm(B), blocks)
