"""B-stationary kernel with more work items than compute units (persistent
workgroups that stage B again for each item) and rows of B and C that are not
aligned for a vector of columns: K = 1024 (every staging register in use), each
type of B, windows with and without sparse parts, items round-robin and by XCD.

Bound per element, with S = sum|a||b| over the row: A and B are rounded to BF16
(2^-9 each) and products added in FP32, so 2^-7 S covers K <= 1024."""
import numpy as np
import pytest
import torch

from stile_amd import _native

from .test_gpu_stream_windows import _operand

pytestmark = pytest.mark.gpu

K = 1024
SIZES = [16, 33, 5, 64, 100, 1, 48, 700] * 8
SPARSE = {False: [0], True: [0, 7, 0, 40, 1]}
_made = {}


def _matrix(mixed):
    if mixed not in _made:
        _made[mixed] = _operand(K, SIZES, SPARSE[mixed], seed=5)
    return _made[mixed]


@pytest.mark.parametrize("b", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("matrices,N,pad", [(1, 4093, 0), (1, 2045, 4), (5, 333, 2), (5, 250, 1)])
def test_more_items_than_compute_units(cuda, b, mixed, matrices, N, pad):
    A, pack = _matrix(mixed)
    M = A.shape[0]
    plan = _native.Plan.spmm([pack] * matrices, "bfloat16")
    plan.set_option("lds_list", 11)  # the most units: one per window here
    assert len(SIZES) * matrices * -(-N // 64) > torch.cuda.get_device_properties(0).multi_processor_count
    rng = np.random.default_rng(N)
    B = torch.full((matrices * K, N + pad), float("nan"), dtype=getattr(torch, b), device=cuda)
    B[:, :N] = torch.from_numpy(rng.uniform(-1, 1, (matrices * K, N)))
    C = torch.full((matrices * M, N + pad), -7.0, device=cuda)
    print("persistent unaligned", b, mixed, matrices, N, pad, flush=True)
    plan.run_spmm(B[:, :N], out=C[:, :N])
    assert torch.all(C[:, N:] == -7.0)
    Ad = torch.from_numpy(A.toarray()).to(cuda)
    for i in range(matrices):
        Bi = B[i * K:(i + 1) * K, :N].double()
        diff = (C[i * M:(i + 1) * M, :N].double() - Ad @ Bi).abs()
        assert torch.all(diff <= 2.0 ** -7 * (Ad.abs() @ Bi.abs())), i
