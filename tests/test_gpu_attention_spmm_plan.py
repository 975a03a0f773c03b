"""stile_attention_run on a plan of stile_plan_create_spmm without dense chunks:
every packed slot is a mask entry, as in a plan made for attention."""
import pytest
import torch

from stile_amd import _native

from .test_gpu_attention_rows import _ell_group, _mask

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blocks", ["float32", "bfloat16"])
@pytest.mark.parametrize("L", [1, 47, 1000])
def test_sparse_only_spmm_plan(cuda, L, blocks):
    mask = _mask(L, [9, 0, 4], L)
    pack = dict(M=L, K=L, ell=[_ell_group(mask.tocoo())], tc=[])
    plan = _native.Plan.spmm(pack, blocks)
    assert plan.info()["num_chunks"] == 0
    plan.attention_plan = True  # the check of the C entry is the one under test
    g = torch.Generator(device=cuda)
    g.manual_seed(L)
    Q, K, V = (torch.randn(L, 64, device=cuda, generator=g).to(torch.bfloat16) for _ in range(3))
    print("attention on an SpMM plan", L, blocks, flush=True)
    got = plan.run_attention(Q, K, V, 0.125)
    assert torch.equal(got, _native.Plan.attention(pack).run_attention(Q, K, V, 0.125))
