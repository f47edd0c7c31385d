"""Pairs grouped by expert (csrc/moe.hip: moe_sort_kernel): one workgroup and several (from 4096 pairs), borders of a thread's pieces of four
and of a workgroup's chunk, one expert for everybody, unused experts, 1 and 512 experts.  Whole numbers: exact; the order inside an
expert's run is free."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,top_k", [(1, 1), (3, 5), (1024, 1), (511, 8), (819, 5), (2047, 2), (2048, 2), (2049, 2), (5003, 3), (8192, 8),
                                          (70001, 3)])
@pytest.mark.parametrize("E,used", [(1, 1), (64, 64), (512, 512), (130, 3)])
def test_pairs_grouped_by_expert(tokens, top_k, E, used):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from nanovllm import ops
    g = torch.Generator().manual_seed(tokens + E)
    ids = (torch.randint(0, used, (tokens, top_k), generator=g) * (E // used)).to(torch.int32)
    offsets, token, index = (t.cpu().long() for t in ops.moe_sort(ids.cuda(), E))
    n = tokens * top_k
    flat = ids.flatten().long()
    assert torch.equal(offsets[:E + 1], torch.cat([torch.zeros(1, dtype=torch.long), torch.bincount(flat, minlength=E).cumsum(0)]))
    assert torch.equal(token[:n], index[:n] // top_k)
    assert torch.equal(flat[index[:n]], flat.sort().values)
    assert torch.equal(index[:n].sort().values, torch.arange(n))
