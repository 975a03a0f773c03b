"""Sparse-only rows and pieces of long rows at the sizes where their kernels can
go wrong: rows of every length around the batch of 8 and the split at 256 (empty
rows and a hub row among them), widths around the 64-column passes, every type
of B, unaligned rows, and a B that 32-bit offsets cannot address.

Bound per element: (n + 2) 2^-24 sum|a||b| for a row of n products, each
rounded once and added in some order in FP32 (or FP64 for long rows)."""
import numpy as np
import pytest
import scipy.sparse
import torch

from stile_amd import _native

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 2, 7, 8, 9, 15, 16, 17, 0, 0, 24, 63, 64, 65, 127, 128, 200, 255, 256, 257, 258, 300, 511, 512, 513,
           1100, 4096, 4097, 0, 5000, 3, 5, 1, 0, 2]


def _matrix(K, seed, lengths=LENGTHS):
    rng = np.random.default_rng(seed)
    cols = [np.sort(rng.choice(K, n, replace=False)) for n in lengths]
    indptr = np.concatenate([[0], np.cumsum([len(c) for c in cols])])
    return scipy.sparse.csr_matrix((rng.uniform(-1, 1, indptr[-1]).astype(np.float32), np.concatenate(cols), indptr),
                                   shape=(len(lengths), K))


def _plan(A):
    """Every nonzero as an ELL tile row of one column, sixteen to a tile (row M: padding)."""
    coo = A.tocoo()
    T = -(-coo.nnz // 16)
    rows, cols = np.full(16 * T, A.shape[0], np.int32), np.zeros(16 * T, np.int32)
    rows[:coo.nnz], cols[:coo.nnz] = coo.row, coo.col
    a, ids = np.zeros(16 * T, np.float32), np.full(16 * T, -1, np.int32)
    a[:coo.nnz], ids[:coo.nnz] = coo.data, np.arange(coo.nnz)
    group = dict(m_blk=16, nnz_cols=1, num_tiles=T, a=a, indices_k=cols, indices_reordered_i=rows, a_ids=ids)
    return _native.Plan.spmm(dict(M=A.shape[0], K=A.shape[1], ell=[group], tc=[]), "float32")


def _check(A, B, C):
    Bd = B.double().cpu().numpy()
    A64 = A.astype(np.float64)
    n = np.diff(A.indptr)[:, None]
    bound = (n + 2) * 2.0 ** -24 * (abs(A64) @ np.abs(Bd))
    diff = np.abs(C.double().cpu().numpy() - A64 @ Bd)
    assert np.all(diff <= bound), (diff - bound).max()
    assert np.all(C.cpu().numpy()[n[:, 0] == 0] == 0)


@pytest.mark.parametrize("N,pad", [(1, 0), (2, 0), (3, 1), (4, 0), (31, 0), (64, 0), (64, 3), (65, 0), (100, 0),
                                   (128, 0), (129, 0), (130, 6), (192, 0), (256, 0), (256, 1), (260, 0), (321, 30)])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16"])
def test_rows_of_every_length_and_width(cuda, N, pad, dtype):
    A = _matrix(6000, 1)
    plan = _plan(A)
    assert plan.info()["num_split"] > 0
    g = torch.Generator(device=cuda)
    g.manual_seed(N)
    B = torch.randn(6000, N + pad, device=cuda, generator=g).to(getattr(torch, dtype))[:, :N]
    print("sparse rows", N, pad, dtype, flush=True)
    _check(A, B, plan.run_spmm(B))
    once, again = plan.run_spmm(B, deterministic=True), plan.run_spmm(B, deterministic=True)
    _check(A, B, once)
    assert torch.equal(once, again)


@pytest.mark.parametrize("rows", [1, 16, 17, 3000])
def test_many_short_rows(cuda, rows):
    rng = np.random.default_rng(rows)
    A = _matrix(500, rows, [int(n) for n in rng.integers(0, 12, rows)])
    plan = _plan(A) if A.nnz else None
    if plan is None:
        A = _matrix(500, rows, [3] * rows)
        plan = _plan(A)
    B = torch.randn(500, 72, device=cuda)
    print("short rows", rows, flush=True)
    _check(A, B, plan.run_spmm(B))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_b_beyond_32_bit_offsets(cuda, dtype):
    K, ld = 700, (1 << 21) if dtype == "float32" else (1 << 22)  # 700 rows of 8 MiB: 5.5 GiB
    A = _matrix(K, 4, [0, 1, 9, 300, 257, 64, 700, 5])
    plan = _plan(A)
    big = torch.empty(K, ld, device=cuda, dtype=getattr(torch, dtype))
    for N in (64, 130, 256):
        B = big[:, :N]
        B.copy_(torch.randn(K, N, device=cuda))
        print("wide B", N, dtype, flush=True)
        _check(A, B, plan.run_spmm(B))


@pytest.mark.parametrize("K", [131072, 131073])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_columns_per_lane_on_both_sides_of_the_b_size_rule(cuda, K, dtype):
    A = _matrix(K, 5, [40] * 1100 + [300, 700, 5000])
    plan = _plan(A)
    g = torch.Generator(device=cuda)
    g.manual_seed(K)
    B = torch.randn(K, 130, device=cuda, generator=g).to(getattr(torch, dtype))
    print("rows", K, dtype, flush=True)
    _check(A, B, plan.run_spmm(B))
    once, again = plan.run_spmm(B, deterministic=True), plan.run_spmm(B, deterministic=True)
    _check(A, B, once)
    assert torch.equal(once, again)
