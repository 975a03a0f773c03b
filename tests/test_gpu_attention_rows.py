"""Fused attention over windows that hold dense chunks, a sparse part, both or
neither: sparse rows around the kernel's step of four entries, row offsets
beyond 32 bits, and scores of -infinity.

Reference: softmax(Q K^T / 8 on the mask) V in float64 on the BF16 inputs.
Bar 1e-2 norm-wise, as for the other BF16 attention tests (probabilities are
rounded to BF16, 2^-9 relative, before they weigh V)."""
import numpy as np
import pytest
import scipy.sparse
import torch

from stile_amd import _native, api, datasets

pytestmark = pytest.mark.gpu


def _reference(mask, Q, K, V):
    q, k, v = (t.double().cpu().numpy() for t in (Q, K, V))
    out = np.zeros_like(q)
    for i in range(mask.shape[0]):
        cols = mask.indices[mask.indptr[i]:mask.indptr[i + 1]]
        if len(cols):
            s = k[cols] @ q[i] / 8
            w = np.exp(s - s.max())
            out[i] = w @ v[cols] / w.sum()
    return out


def _mask(L, counts, seed):
    """Row i holds counts[i % len(counts)] distinct columns; every 32nd window is a band too."""
    rng = np.random.default_rng(seed)
    rows, cols = [], []
    for i in range(L):
        c = rng.choice(L, min(L, counts[i % len(counts)]), replace=False)
        rows += [i] * len(c)
        cols += list(c)
    m = scipy.sparse.csr_matrix((np.ones(len(rows), np.float32), (rows, cols)), shape=(L, L))
    m.sort_indices()
    return m


def _ell_group(coo):
    """Every entry as an ELL tile row of one column, sixteen to a tile (row L: padding)."""
    T = -(-coo.nnz // 16)
    rows, cols = np.full(16 * T, coo.shape[0], np.int32), np.zeros(16 * T, np.int32)
    rows[:coo.nnz], cols[:coo.nnz] = coo.row, coo.col
    a, ids = np.zeros(16 * T, np.float32), np.full(16 * T, -1, np.int32)
    a[:coo.nnz], ids[:coo.nnz] = coo.data, np.arange(coo.nnz)
    return dict(m_blk=16, nnz_cols=1, num_tiles=T, a=a, indices_k=cols, indices_reordered_i=rows, a_ids=ids)


def _plan(mask, dense):
    """dense: the band |i - j| < 24 in TC tiles and the other entries sparse; else all sparse."""
    coo = mask.tocoo()
    near = np.abs(coo.row - coo.col) < (24 if dense else 0)
    parts = [scipy.sparse.coo_matrix((coo.data[s], (coo.row[s], coo.col[s])), shape=mask.shape) for s in (near, ~near)]
    tc = api.spmm_pack(parts[0].tocsr(), api.SearchOptions(only_TC=True))[0]["tc"] if dense else []
    return _native.Plan.attention(dict(M=mask.shape[0], K=mask.shape[1], ell=[_ell_group(parts[1])], tc=tc))


@pytest.mark.parametrize("L,counts,dense", [(16, [1], False), (47, [0, 1, 3, 4, 5], False),
                                            (100, [8, 7, 9, 0, 31, 2, 64], False), (257, [4, 5, 40], True),
                                            (1000, [12, 3, 1], True)])
def test_rows_of_every_length(cuda, L, counts, dense):
    mask = _mask(L, counts, L)
    if dense:
        mask = ((mask + datasets.attention_mask(L, band=40, n_random=0)) > 0).astype(np.float32).tocsr()
        mask.sort_indices()
    plan = _plan(mask, dense)
    info = plan.info()
    assert info["sparse_nnz"] > 0 and (info["num_chunks"] > 0) == dense
    g = torch.Generator(device=cuda)
    g.manual_seed(L)
    big = torch.randn(L, 3 * 64 + 8, device=cuda, generator=g).to(torch.bfloat16)  # leading dimension 200
    Q, K, V = (big[:, 64 * i:64 * i + 64] for i in range(3))
    print("attention rows", L, counts, dense, flush=True)
    got = plan.run_attention(Q, K, V, 0.125).double().cpu().numpy()
    ref = _reference(mask, Q, K, V)
    assert np.max(np.abs(got - ref)) <= 1e-2 * np.max(np.abs(ref))
    empty = np.diff(mask.indptr) == 0
    assert np.all(got[empty] == 0)


def test_row_offsets_beyond_32_bits(cuda):
    L, ld = 264, 1 << 23  # 264 rows of 16 MiB: 4.1 GiB
    mask = ((_mask(L, [9, 2], 5) + datasets.attention_mask(L, band=40, n_random=0)) > 0).astype(np.float32).tocsr()
    mask.sort_indices()
    plan = _plan(mask, True)
    big = torch.empty(L, ld, device=cuda, dtype=torch.bfloat16)
    g = torch.Generator(device=cuda)
    g.manual_seed(1)
    big[:, :192] = torch.randn(L, 192, device=cuda, generator=g).to(torch.bfloat16)
    Q, K, V = (big[:, 64 * i:64 * i + 64] for i in range(3))
    print("attention wide rows", flush=True)
    got = plan.run_attention(Q, K, V, 0.125).double().cpu().numpy()
    ref = _reference(mask, Q, K, V)
    assert np.max(np.abs(got - ref)) <= 1e-2 * np.max(np.abs(ref))


def test_scores_of_minus_infinity_weigh_nothing(cuda):
    """A key of -infinity against positive queries scores -infinity: it gets
    no weight, and a row with only such keys is 0."""
    L = 64
    mask = _mask(L, [6], 3)
    plan = _plan(mask, False)
    g = torch.Generator(device=cuda)
    g.manual_seed(2)
    Q, K, V = (torch.rand(L, 64, device=cuda, generator=g).to(torch.bfloat16) + 0.5 for _ in range(3))
    dead = np.zeros(L, bool)
    dead[mask.indices[:mask.indptr[1]]] = True  # every key of row 0
    K[torch.from_numpy(dead).to(cuda)] = float("-inf")
    print("attention -inf keys", flush=True)
    got = plan.run_attention(Q, K, V, 0.125).double().cpu().numpy()
    left = scipy.sparse.csr_matrix(mask.toarray() * ~dead[None, :])
    ref = _reference(left, Q, K.nan_to_num(neginf=0.0), V)
    assert np.all(got[0] == 0)
    assert np.max(np.abs(got - ref)) <= 1e-2 * np.max(np.abs(ref))
