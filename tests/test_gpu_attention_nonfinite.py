"""Fused attention when V holds infinities or NaN: a row whose entries do not
reach them comes out as if they were not there."""
import numpy as np
import pytest
import scipy.sparse
import torch

from stile_amd import _native

from .test_gpu_attention_rows import _ell_group, _mask

pytestmark = pytest.mark.gpu


def _sparse_plan(masks):
    return _native.Plan.attention([dict(M=m.shape[0], K=m.shape[1], ell=[_ell_group(m.tocoo())], tc=[]) for m in masks])


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("counts", [[5], [4, 1, 7], [0, 3, 8]])
def test_rows_that_do_not_reach_them_stay_as_they_are(cuda, bad, counts):
    L = 100
    masks = [_mask(L, counts, s) for s in (1, 2)]  # two sequences: rows 0 .. L - 1 and L .. 2L - 1
    plan = _sparse_plan(masks)
    both = scipy.sparse.block_diag(masks).tocsr()
    g = torch.Generator(device=cuda)
    g.manual_seed(4)
    Q, K, V = (torch.randn(2 * L, 64, device=cuda, generator=g).to(torch.bfloat16) for _ in range(3))
    print("attention non-finite V", bad, counts, flush=True)
    before = plan.run_attention(Q, K, V, 0.125)
    for row in (0, L - 1, L):
        W = V.clone()
        W[row] = bad
        got = plan.run_attention(Q, K, W, 0.125)
        hit = torch.from_numpy(np.asarray((both[:, [row]] != 0).todense()).ravel()).to(cuda)
        assert torch.equal(got[~hit], before[~hit])
        assert not torch.isfinite(got[hit]).any()
