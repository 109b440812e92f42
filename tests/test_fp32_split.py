"""The fp32 kernel's last round, cut along the reduction: operands of small integers, whose sums are exact in any order, so the
product has to equal the exact one bit for bit, launch after launch (the exchange memory is reused)."""

import pytest
import torch

from flash_model_architectures_amd import ops
from oracle import torch_oracle as to

from .helpers import TOL, assert_close, gemm_form


# rows per expert, columns, reduction, rows of the tiles; 2, 3 and 8 parts of 128-row tiles, 4 of 64-row ones, 8 of 32-row ones
CASES = [
    ([1024, 1, 2050, 1100], 2048, 1216, 128),
    ([1024, 1, 2050, 1100], 2040, 2004, 128),
    ([1024, 0, 2050, 1100], 2048, 4100, 128),
    ([700, 1, 1300, 1000], 2048, 4100, 64),
    ([350, 1, 650, 500], 256, 28000, 32),
]


@pytest.mark.gpu
@pytest.mark.parametrize("sizes,N,K,height", CASES)
@pytest.mark.parametrize("form", ["TN", "TN+swiglu", "NN", "NN+swiglu_bwd"])
def test_exact_sums(form, sizes, N, K, height):
    dev = "cuda"
    E, M = len(sizes), sum(sizes)
    kind, epilogue = form[:2], {"TN+swiglu": 1, "NN+swiglu_bwd": 2}.get(form, 0)
    assert gemm_form(kind, torch.float32, E, M, N, K, epilogue) == ("tiled", height, 128)
    g = torch.Generator(dev).manual_seed(K)
    ends = torch.tensor(sizes).cumsum(0).tolist()
    offsets = torch.tensor([0] + ends, dtype=torch.int32, device=dev)
    rows = [slice(end - size, end) for end, size in zip(ends, sizes)]
    index = torch.randperm(M, generator=g, device=dev).int()
    saved = torch.randn(M, 2 * N, generator=g, device=dev)
    for _ in range(2):
        a = torch.randint(-2, 3, (M, K), generator=g, device=dev).float()
        w = torch.randint(-1, 2, (E, K, N), generator=g, device=dev).float()
        want = torch.cat([(a[r].double() @ w[e].double()).float() for e, r in enumerate(rows)])
        stored = w.transpose(1, 2).contiguous()  # [E, N, K]
        for _ in range(2):
            out = torch.full((M, N), float("nan"), device=dev)
            if form == "TN+swiglu":
                act = torch.full((M, N // 2), float("nan"), device=dev)
                x = torch.empty_like(a)
                x[index.long()] = a
                ops.up_projection_fused(x, stored, index, offsets, act, out, 1, "swiglu")
                assert torch.equal(out, want)
                assert_close(act, to.swiglu_packed(want), TOL[torch.float32], "activation of a split tile")
            elif form == "NN+swiglu_bwd":
                d_pre = torch.full((M, 2 * N), float("nan"), device=dev)
                ops.down_projection_dgrad_fused(a, w, saved, offsets, d_pre, "swiglu")
                leaf = saved.double().requires_grad_()
                to.swiglu_packed(leaf).backward(want.double())
                assert_close(d_pre, leaf.grad.float(), TOL[torch.float32], "activation backward of a split tile")
            else:
                weights = stored.permute(0, 2, 1) if kind == "TN" else w
                ops.scatter2scatter(a, weights, index, index, out, 1, True, False, offsets)
                assert torch.equal(out[index.long()], want)
