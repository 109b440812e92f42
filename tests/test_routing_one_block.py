"""The counting sort of up to 4096 ids in one block, at the edges of its waves' runs and of its scan over the experts."""

import pytest
import torch

import flash_model_architectures_amd as xma


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("experts", [1, 2, 63, 64, 65, 129, 512])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025, 2049, 4095, 4096, 4097])
def test_one_block(n, experts, dtype):
    g = torch.Generator().manual_seed(n + experts)
    uniform = torch.randint(0, experts, (n,), generator=g)
    for ids in (uniform, torch.full((n,), experts - 1), (uniform * uniform) // experts):
        r = xma.route_tokens(ids.to(dtype).cuda(), experts)
        counts = torch.bincount(ids, minlength=experts)
        order = torch.argsort(ids, stable=True)
        assert torch.equal(r.expert_frequency.cpu().long(), counts)
        assert torch.equal(r.expert_offsets.cpu().long(), torch.cat([torch.zeros(1, dtype=torch.long), counts.cumsum(0)]))
        assert torch.equal(r.sorted_scattered_idxs.cpu().long(), order)
        assert torch.equal(r.sorted_expert_idxs.cpu().long(), ids[order])
