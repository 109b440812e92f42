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


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize(
    "tokens,experts,k",
    [
        (1, 1, 1), (1, 64, 6), (3, 512, 1), (31, 7, 3), (64, 64, 6), (128, 64, 6), (129, 64, 6), (512, 8, 2), (513, 8, 2), (1024, 8, 1),
        (1025, 8, 1), (5, 300, 5), (5, 512, 6), (17, 600, 2), (40, 128, 8),
    ],
)  # fmt: skip
def test_selection_and_routing_in_one_launch(tokens, experts, k, dtype):
    """`xma_topk_route` on both sides of the lines up to which one block does it all, against the two entry points."""

    from flash_model_architectures_amd import _native

    g = torch.Generator("cuda").manual_seed(tokens)
    logits = torch.randn(tokens, experts, generator=g, device="cuda").to(dtype)
    logits[0] = 0.25  # ties
    if tokens > 2:
        logits[1], logits[2, 0] = float("-inf"), float("nan")
    weights, selected = xma.topk_softmax(logits, k)
    routing = xma.route_tokens(selected, experts)

    def empty(*shape, kind=torch.int32):
        return torch.empty(shape, dtype=kind, device="cuda")

    w, s = empty(tokens, k, kind=dtype), empty(tokens, k, kind=torch.int64)
    counts, offsets, ids, perm = empty(experts), empty(experts + 1), empty(tokens * k), empty(tokens * k)
    workspace = empty(1 << 20, kind=torch.uint8)
    _native.call(
        "xma_topk_route", logits.data_ptr(), _native.dtype_code(logits), tokens, experts, k, experts, w.data_ptr(), s.data_ptr(),
        counts.data_ptr(), offsets.data_ptr(), ids.data_ptr(), perm.data_ptr(), workspace.data_ptr(), workspace.numel(),
        _native.stream(),
    )  # fmt: skip
    assert torch.equal(w.view(torch.uint8), weights.view(torch.uint8)) and torch.equal(s, selected)
    assert torch.equal(counts, routing.expert_frequency.view(torch.int32)) and torch.equal(offsets, routing.expert_offsets)
    assert torch.equal(ids, routing.sorted_expert_idxs) and torch.equal(perm, routing.sorted_scattered_idxs)
