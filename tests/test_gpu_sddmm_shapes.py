"""SDDMM at the feature counts, strides and entry counts where its kernel can go
wrong: 1D entries around the group of four and the lanes per entry, dense blocks
below and above the features from which four waves share one, unaligned rows and
operands that 32-bit offsets cannot address.

Bound per element: (Kf + 2) 2^-24 sum|x||y| (Kf products, each rounded once and
added in FP32 in some order)."""
import numpy as np
import pytest
import torch

from stile_amd import _native

pytestmark = pytest.mark.gpu


def _pack(M, N, n1d, nblk, seed):
    """n1d single entries (sorted by row) and nblk dense 16 x 16 blocks, each
    output once; returns (rows, cols, pack)."""
    rng = np.random.default_rng(seed)
    r1 = np.sort(rng.integers(0, M, n1d))
    c1 = rng.integers(0, N, n1d)
    br = np.stack([rng.choice(M, 16, replace=False) for _ in range(nblk)]) if nblk else np.zeros((0, 16), int)
    bc = np.stack([rng.choice(N, 16, replace=False) for _ in range(nblk)]) if nblk else np.zeros((0, 16), int)
    pos = [np.sort(rng.choice(256, rng.integers(1, 257), replace=False)) for _ in range(nblk)]
    indptr = np.concatenate([[0], np.cumsum([len(q) for q in pos])]).astype(np.int32)
    allpos = np.concatenate(pos) if nblk else np.zeros(0, int)
    b = np.repeat(np.arange(nblk), np.diff(indptr))
    rows = np.concatenate([r1, br[b, allpos // 16]])
    cols = np.concatenate([c1, bc[b, allpos % 16]])
    ids = rng.permutation(len(rows))  # the output of each entry
    g1d = [dict(mid_idx=r1, j_idx=c1, remap=ids[:n1d])] if n1d else []
    tc = [dict(nnzb=nblk, blk_k=16, i_indices=br, j_indices=bc, indptr=indptr, indices_dense=allpos,
               indices=ids[n1d:])] if nblk else []
    out_r, out_c = np.empty_like(rows), np.empty_like(cols)
    out_r[ids], out_c[ids] = rows, cols
    return out_r, out_c, dict(M=M, N=N, nnz=len(rows), g1d=g1d, tc=tc)


def _check(rows, cols, X, Y, out):
    x, y = X.double().cpu().numpy()[rows], Y.double().cpu().numpy()[cols]
    bound = (X.shape[1] + 2) * 2.0 ** -24 * (np.abs(x) * np.abs(y)).sum(1)
    assert np.all(np.abs(out.double().cpu().numpy() - (x * y).sum(1)) <= bound)


@pytest.mark.parametrize("Kf", [1, 2, 3, 4, 5, 7, 8, 12, 16, 20, 31, 32, 33, 48, 63, 64, 65, 100, 127, 128, 131, 192,
                                256, 300, 1024])
@pytest.mark.parametrize("pad", [0, 3, 4])
@pytest.mark.parametrize("n1d,nblk", [(1, 0), (7, 3), (0, 1), (4001, 37)])
def test_feature_counts(cuda, Kf, pad, n1d, nblk):
    rows, cols, pack = _pack(200, 300, n1d, nblk, Kf + n1d)
    plan = _native.Plan.sddmm(pack)
    g = torch.Generator(device=cuda)
    g.manual_seed(Kf)
    X = torch.randn(200, Kf + pad, device=cuda, generator=g)[:, :Kf]
    Y = torch.randn(300, Kf + pad, device=cuda, generator=g)[:, :Kf]
    if pad:  # what lies between the rows takes no part
        for t in (X, Y):
            torch.as_strided(t, (t.shape[0], pad), (Kf + pad, 1), Kf).fill_(float("nan"))
    print("sddmm", Kf, pad, n1d, nblk, flush=True)
    _check(rows, cols, X, Y, plan.run_sddmm(X, Y))


@pytest.mark.parametrize("Kf", [64, 130])
def test_operands_beyond_32_bit_offsets(cuda, Kf):
    rows, cols, pack = _pack(300, 100, 1000, 20, 3)
    plan = _native.Plan.sddmm(pack)
    X = torch.empty(300, 1 << 22, device=cuda)[:, :Kf]  # rows of 16 MiB: 5 GB
    X.copy_(torch.randn(300, Kf, device=cuda))
    Y = torch.randn(100, Kf, device=cuda)
    print("sddmm wide rows", Kf, flush=True)
    _check(rows, cols, X, Y, plan.run_sddmm(X, Y))
