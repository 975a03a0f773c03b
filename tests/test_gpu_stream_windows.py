"""Streaming kernel (FP32 and FP16 blocks, BF16 blocks with K > 1024) at the
window shapes where it can go wrong: 1 to 20 chunks around the shares of its
waves and the change to 32 columns a workgroup, a huge window cut into parts,
sparse parts of 0 to 300 entries per row on both sides of the fold, widths
around its 32- and 64-column blocks, unaligned rows and a B that 24-bit row
offsets cannot address.

Bounds per element, with S = sum|a||b| over the row: FP32 (n + 2) 2^-23 S for n
products (each rounded once, added in FP32); 16-bit blocks 2^-7 S (A and B
rounded to BF16, 2^-9 each, or FP16, less)."""
import numpy as np
import pytest
import scipy.sparse
import torch

from stile_amd import _native

pytestmark = pytest.mark.gpu


def _operand(K, cols_per_window, sparse_per_row, seed):
    """A CSR matrix of 16-row windows: window w holds cols_per_window[w] full
    columns (TC tiles of 16 columns) and its row r sparse_per_row[(16 w + r) %
    len] more entries (ELL); returns (matrix, pack)."""
    rng = np.random.default_rng(seed)
    M = 16 * len(cols_per_window)
    tc_a, tc_cols, indptr, er, ec, ev = [], [], [0], [], [], []
    dense = {}
    for w, n in enumerate(cols_per_window):
        pick = rng.permutation(K)
        cols, rest = np.sort(pick[:n]), pick[n:]
        for t in range(0, n, 16):
            c = cols[t:t + 16]
            a = np.zeros((16, 16), np.float32)
            a[:, :len(c)] = rng.uniform(-1, 1, (16, len(c)))
            tc_a.append(a)
            tc_cols.append(np.concatenate([c, np.full(16 - len(c), c[0])]))
            for j, cc in enumerate(c):
                for r in range(16):
                    dense[16 * w + r, cc] = a[r, j]
        indptr.append(len(tc_a))
        for r in range(16):
            s = sparse_per_row[(16 * w + r) % len(sparse_per_row)]
            er += [16 * w + r] * s
            ec += list(rest[:s])
            ev += list(rng.uniform(-1, 1, s))
    T = -(-max(len(er), 1) // 16)
    rows, cols, vals = np.full(16 * T, M, np.int32), np.zeros(16 * T, np.int32), np.zeros(16 * T, np.float32)
    rows[:len(er)], cols[:len(er)], vals[:len(er)] = er, ec, ev
    ell = [dict(m_blk=16, nnz_cols=1, num_tiles=T, a=vals, indices_k=cols, indices_reordered_i=rows)] if er else []
    tc = [dict(group_size=16, num_windows=len(cols_per_window), nnzb=len(tc_a), rows_2d=False, k_notsorted=False,
               a=np.stack(tc_a), i_indices=np.arange(len(cols_per_window)), indptr=np.array(indptr),
               indices=np.stack(tc_cols))]
    keys = list(dense) + list(zip(er, ec))
    A = scipy.sparse.csr_matrix((np.concatenate([list(dense.values()), vals[:len(er)]]).astype(np.float64),
                                 ([k[0] for k in keys], [k[1] for k in keys])), shape=(M, K))
    return A, dict(M=M, K=K, ell=ell, tc=tc)


def _check(A, B, C, blocks):
    Bd = B.double().cpu().numpy()
    S = abs(A) @ np.abs(Bd)
    n = np.diff(A.indptr)[:, None]
    bound = (n + 2) * 2.0 ** -23 * S if blocks == "float32" else 2.0 ** -7 * S
    diff = np.abs(C.double().cpu().numpy() - A @ Bd)
    assert np.all(diff <= bound), float((diff / np.maximum(S, 1e-30)).max())


WINDOWS = [1, 16, 31, 32, 33, 64, 255, 256, 257, 300, 500, 513, 544, 600, 5, 700]


@pytest.mark.parametrize("blocks,b", [("float32", "float32"), ("float32", "bfloat16"), ("float16", "float16"),
                                      ("float16", "float32"), ("float16", "bfloat16"), ("bfloat16", "bfloat16"),
                                      ("bfloat16", "float32"), ("bfloat16", "float16")])
@pytest.mark.parametrize("N,pad", [(1, 0), (9, 0), (32, 0), (33, 0), (64, 0), (65, 3), (100, 0), (128, 0), (321, 30)])
@pytest.mark.parametrize("sparse", [[0], [0, 3, 0, 0, 17, 128], [0, 5, 129, 300]])
def test_window_shapes(cuda, blocks, b, N, pad, sparse):
    A, pack = _operand(1300, WINDOWS, sparse, len(sparse))
    plan = _native.Plan.spmm(pack, blocks)
    g = torch.Generator(device=cuda)
    g.manual_seed(N)
    B = torch.randn(1300, N + pad, device=cuda, generator=g).to(getattr(torch, b))[:, :N]
    print("stream", blocks, b, N, pad, sparse, flush=True)
    _check(A, B, plan.run_spmm(B), blocks)
    once, again = plan.run_spmm(B, deterministic=True), plan.run_spmm(B, deterministic=True)
    _check(A, B, once, blocks)
    assert torch.equal(once, again)


@pytest.mark.parametrize("blocks", ["float32", "bfloat16"])
def test_huge_window_and_many_small_ones(cuda, blocks):
    A, pack = _operand(9000, [8700] + [20, 40] * 300, [0, 2], 7)
    plan = _native.Plan.spmm(pack, blocks)
    B = torch.randn(9000, 96, device=cuda)
    print("stream huge", blocks, flush=True)
    _check(A, B, plan.run_spmm(B), blocks)
    once, again = plan.run_spmm(B, deterministic=True), plan.run_spmm(B, deterministic=True)
    _check(A, B, once, blocks)
    assert torch.equal(once, again)


@pytest.mark.parametrize("blocks,b", [("float32", "float32"), ("bfloat16", "bfloat16")])
def test_rows_beyond_24_bit_offsets(cuda, blocks, b):
    ld = 1 << 23  # 2^24 bytes and more per row, 1100 rows: 18 / 35 GB
    A, pack = _operand(1100, [40, 300, 600], [0, 4], 9)
    plan = _native.Plan.spmm(pack, blocks)
    B = torch.empty(1100, ld, device=cuda, dtype=getattr(torch, b))[:, :70]
    B.copy_(torch.randn(1100, 70, device=cuda))
    print("stream wide rows", blocks, flush=True)
    _check(A, B, plan.run_spmm(B), blocks)
