"""Products whose workgroups are more than one launch takes (a grid dimension holds
fewer than 2^32 threads): few rows and 2^22 columns, so that the matrices stay small.

Every entry of C is written; columns at the ends, at the cuts and between are
compared with FP64, per element within (n + 2) 2^-24 sum|a||b| for rows of n
entries (n products, rounded and added in FP32 in some order), 2^-7 sum|a||b|
for BF16 blocks (A rounded to BF16, 2^-9, the sums as above)."""
import numpy as np
import pytest
import scipy.sparse
import torch

from stile_amd import _native, api

pytestmark = pytest.mark.gpu

N = 1 << 22


def _run(cuda, A, search, deterministic, blocks="float32", N=N):
    opts = api.options_for(blocks)
    setattr(opts, search, True)
    plan = _native.Plan.spmm(api.spmm_pack(A, opts)[0], blocks)
    g = torch.Generator(device=cuda)
    g.manual_seed(1)
    B = torch.randn(A.shape[1], N, device=cuda, generator=g, dtype=getattr(torch, blocks))
    C = torch.full((A.shape[0], N), float("nan"), device=cuda)
    print("launch limits", A.shape, A.nnz, search, deterministic, plan.info(), flush=True)
    plan.run_spmm(B, C, deterministic=deterministic)
    for r in range(0, A.shape[0], 128):
        assert not torch.isnan(C[r:r + 128]).any()
    cols = torch.cat([torch.arange(130), torch.arange(N // 2 - 70, N // 2 + 70), torch.arange(N - 130, N),
                      torch.randint(N, (200,), generator=torch.Generator().manual_seed(2))]).to(cuda)
    A64, B64 = torch.from_numpy(A.toarray()).to(cuda).double(), B[:, cols].double()
    unit = (np.diff(A.indptr).max() + 2) * 2.0 ** -24 if blocks == "float32" else 2.0 ** -7
    bound = unit * (A64.abs() @ B64.abs())
    assert torch.all((C[:, cols].double() - A64 @ B64).abs() <= bound)
    return plan.info()


@pytest.fixture(autouse=True)
def _free(cuda):
    yield
    torch.cuda.empty_cache()


def _full(M, K):
    return scipy.sparse.csr_matrix(np.random.default_rng(M + K).standard_normal((M, K)).astype(np.float32))


def test_sparse_rows(cuda):
    # 2048 wave tasks of 24 and 96 entries in turn, 32768 column chunks of 128
    A = _full(2048, 96).toarray()
    A[::2, 24:] = 0
    info = _run(cuda, scipy.sparse.csr_matrix(A), "only_ELL", False)
    assert info["num_chunks"] == 0 and info["num_split"] == 0


def test_even_rows(cuda):
    # 16384 rows of 64 entries, four to a wave, 16384 column chunks of 64 (2^20 columns)
    info = _run(cuda, _full(16384, 64), "only_ELL", False, N=1 << 20)
    assert info["num_chunks"] == 0 and info["num_split"] == 0


@pytest.mark.parametrize("deterministic", [False, True])
def test_pieces_of_long_rows(cuda, deterministic):
    # 512 pieces behind 256 rows' first 256 entries, 32768 column chunks of 128;
    # the reduce kernel 256 rows of 65536 chunks of 64
    info = _run(cuda, _full(256, 768), "only_ELL", deterministic)
    assert info["num_split"] == 512


def test_dense_windows(cuda):
    # 128 windows of 6 chunks, a workgroup for each 64 of 2^22 columns
    info = _run(cuda, _full(2048, 192), "only_TC", False)
    assert info["sparse_nnz"] == 0 and info["num_chunks"] == 768


@pytest.mark.parametrize("deterministic", [False, True])
def test_parts_of_huge_windows(cuda, deterministic):
    # 64 windows of 257 chunks in two parts each, a workgroup for each 32 of 2^21 columns
    info = _run(cuda, _full(1024, 8224), "only_TC", deterministic, "bfloat16", 1 << 21)
    assert info["num_chunks"] == 64 * 257
