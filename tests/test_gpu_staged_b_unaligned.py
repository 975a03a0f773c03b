"""B-stationary kernel (BF16 blocks, K <= 1024) where rows of B and C are not
aligned for a vector of columns: widths below one 16-byte piece, around its 4,
8 and 64 columns, odd leading dimensions and bases, each type of B, one matrix
and a batch of two (with rows that hold dense and sparse parts).  Columns past N
of a padded C stay as they were.

Bound per element, with S = sum|a||b| over the row: A and B are rounded to BF16
(2^-9 each) and products added in FP32, so 2^-7 S covers K <= 1024."""
import numpy as np
import pytest
import torch

from stile_amd import _native
from .test_gpu_stream_windows import _operand

pytestmark = pytest.mark.gpu

K = 200
A, PACK = _operand(K, [16, 33, 5, 64, 100, 1], [0, 7, 40], seed=3)
WIDTHS = [1, 2, 3, 4, 5, 7, 8, 9, 11, 15, 33, 61, 62, 63, 64, 65, 68, 101, 129, 333]


def _padded(rows, N, ld, shift, dtype, fill):
    """A (rows, N) view with leading dimension ld whose base is `shift` elements
    past an allocation's start."""
    flat = torch.full((rows * ld + shift,), fill, dtype=dtype, device="cuda:0")
    return flat, flat[shift:].view(rows, ld)[:, :N]


@pytest.mark.parametrize("b", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("pad,shift", [(0, 0), (1, 0), (3, 1), (7, 3)])
@pytest.mark.parametrize("matrices", [1, 2])
def test_unaligned_rows(cuda, b, pad, shift, matrices):
    plan = _native.Plan.spmm([PACK] * matrices if matrices > 1 else PACK, "bfloat16")
    rng = np.random.default_rng(7)
    for N in WIDTHS:
        ld = N + pad
        _, B = _padded(matrices * K, N, ld, shift, getattr(torch, b), float("nan"))
        B.copy_(torch.from_numpy(rng.uniform(-1, 1, B.shape)))
        flat, C = _padded(matrices * A.shape[0], N, ld, shift, torch.float32, -7.0)
        print("unaligned", b, pad, shift, matrices, N, flush=True)
        plan.run_spmm(B, out=C)
        Bd = B.double().cpu().numpy()
        for i in range(matrices):
            Bi = Bd[i * K:(i + 1) * K]
            got = C[i * A.shape[0]:(i + 1) * A.shape[0]].double().cpu().numpy()
            diff, bound = np.abs(got - A @ Bi), 2.0 ** -7 * (abs(A) @ np.abs(Bi))
            assert np.all(diff <= bound), (N, i)
        C.fill_(-7.0)
        assert torch.all(flat == -7.0), N
