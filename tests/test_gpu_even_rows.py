"""Sparse-only rows of much the same lengths (one row per 16-lane group): lengths
around the kernel's steps of eight entries, a last window that is not full, widths
around its 64-column chunks, padded rows, rows that end in an infinity.

Bound per element: (n + 2) 2^-24 sum|a||b| for rows of n entries (n products, each
rounded once and added in FP32 in some order)."""
import numpy as np
import pytest
import scipy.sparse
import torch

from stile_amd import _native, api

pytestmark = pytest.mark.gpu


def _matrix(M, K, lens, seed):
    rng = np.random.default_rng(seed)
    n = np.array([lens[i % len(lens)] for i in range(M)])
    cols = np.concatenate([np.sort(rng.choice(K, c, replace=False)) for c in n])
    A = scipy.sparse.csr_matrix((rng.uniform(-1, 1, len(cols)).astype(np.float32), cols,
                                 np.concatenate([[0], np.cumsum(n)])), shape=(M, K))
    opts = api.options_for("float32")
    opts.only_ELL = True
    return A, _native.Plan.spmm(api.spmm_pack(A, opts)[0], "float32")


LENS = {"short": [16, 17, 18, 15], "steps": [24, 23, 25, 22, 24, 21], "equal": [32], "long": [250, 256, 249, 255]}


@pytest.mark.parametrize("lens", list(LENS))
@pytest.mark.parametrize("M,N,pad", [(8203, 128, 0), (8203, 100, 4), (8203, 68, 8), (5000, 256, 0), (3000, 508, 4)])
def test_even_rows(cuda, lens, M, N, pad):
    A, plan = _matrix(M, 700, LENS[lens], M + N)
    g = torch.Generator(device=cuda)
    g.manual_seed(N)
    B = torch.full((700, N + pad), float("nan"), device=cuda)
    B[:, :N] = torch.randn(700, N, device=cuda, generator=g)
    C = torch.full((M, N + pad), 7.0, device=cuda)
    print("even rows", lens, M, N, pad, flush=True)
    plan.run_spmm(B[:, :N], C[:, :N])
    assert torch.all(C[:, N:] == 7.0)
    A64, B64 = torch.from_numpy(A.toarray()).to(cuda).double(), B[:, :N].double()
    bound = (np.diff(A.indptr).max() + 2) * 2.0 ** -24 * (A64.abs() @ B64.abs())
    assert torch.all((C[:, :N].double() - A64 @ B64).abs() <= bound)
    # an infinity in a B row reaches the rows that hold its column and no others
    W = B.clone()
    W[int(A.indices[A.indptr[1] - 1])] = float("inf")
    D = plan.run_spmm(W[:, :N])
    hit = torch.from_numpy(np.asarray((A[:, [int(A.indices[A.indptr[1] - 1])]] != 0).todense()).ravel()).to(cuda)
    assert torch.equal(D[~hit], C[:, :N][~hit])
    assert torch.isinf(D[hit]).all()
