"""Which kernel and tile the grouped GEMM takes, at both sides of every line that its rules draw (no GPU needed)."""

import pytest
import torch

from .helpers import gemm_form

BF16, FP32 = torch.bfloat16, torch.float32
SWIGLU = 1


@pytest.mark.parametrize(
    "dtype,experts,rows,n,k,form",
    [
        # one tile per expert; then taller tiles the more rows there are, so that a skewed call has few of them
        (BF16, 128, 16, 1536, 2048, ("streaming", 16, 32)),
        (BF16, 128, 17, 1536, 2048, ("streaming", 32, 32)),
        (BF16, 128, 511, 1536, 2048, ("streaming", 32, 32)),
        (BF16, 128, 512, 1536, 2048, ("streaming", 32, 64)),
        (BF16, 128, 1024, 1536, 2048, ("streaming", 32, 64)),
        (BF16, 128, 1025, 1536, 2048, ("streaming", 64, 64)),
        (BF16, 128, 5120, 1536, 2048, ("streaming", 64, 64)),
        (BF16, 128, 5121, 1536, 2048, ("tiled", 256, 256)),
        # short reductions
        (BF16, 128, 511, 2048, 768, ("streaming", 16, 32)),
        (BF16, 128, 512, 2048, 768, ("streaming", 32, 64)),
        (BF16, 128, 2560, 2048, 768, ("streaming", 32, 64)),
        (BF16, 128, 2561, 2048, 768, ("tiled", 256, 256)),
        (BF16, 64, 300, 2048, 1016, ("streaming", 16, 32)),
        (BF16, 64, 300, 2048, 1024, ("streaming", 32, 32)),
        (BF16, 64, 2560, 1024, 2040, ("streaming", 64, 64)),  # 256 tiles of 256 x 256 when every expert has one
        (BF16, 64, 2560, 1032, 2040, ("tiled", 256, 256)),
        # many columns
        (BF16, 8, 16, 28672, 4096, ("streaming", 16, 64)),
        (BF16, 8, 64, 28672, 4096, ("streaming", 32, 64)),
        (BF16, 8, 160, 28672, 4096, ("streaming", 64, 64)),
        (BF16, 8, 161, 28672, 4096, ("streaming", 64, 128)),
        (BF16, 8, 161, 16368, 4096, ("streaming", 64, 64)),
        # the longest reductions
        (BF16, 8, 160, 4096, 14336, ("streaming", 64, 64)),
        (BF16, 8, 161, 4096, 8192, ("streaming", 64, 64)),
        (BF16, 8, 161, 4096, 8200, ("tiled", 256, 256)),
        (BF16, 8, 161, 16384, 8200, ("streaming", 64, 128)),
        # fp32: beyond eight rows per expert only where the tiles do not fill the device
        (FP32, 64, 16, 2048, 2048, ("streaming", 16, 32)),
        (FP32, 64, 512, 2048, 2048, ("streaming", 32, 32)),
        (FP32, 64, 513, 2048, 2048, ("tiled", 32, 128)),
        (FP32, 64, 1536, 2048, 2048, ("tiled", 32, 128)),
        (FP32, 8, 192, 2048, 8192, ("streaming", 32, 64)),
        (FP32, 8, 193, 2048, 8192, ("tiled", 32, 128)),
        # more experts than a wave looks up; not whole vectors
        (BF16, 513, 600, 2048, 2048, ("tiled", 256, 256)),
        (BF16, 8, 64, 2048, 2044, ("element-wise", 128, 128)),
        (FP32, 8, 64, 2046, 2048, ("element-wise", 64, 128)),
    ],
)
def test_forward_forms(dtype, experts, rows, n, k, form):
    got = gemm_form("TN", dtype, experts, rows, n, k)
    assert got[0] == form[0] and (form[0] == "element-wise" or got == form)


def test_gated_columns_pair_whole_chunks():
    assert gemm_form("TN", BF16, 8, 64, 2064, 2048, SWIGLU)[0] == "streaming"
    assert gemm_form("TN", BF16, 8, 64, 2056, 2048, SWIGLU)[0] == "element-wise"
    assert gemm_form("TN", BF16, 8, 64, 2056, 2048)[0] == "streaming"


def test_other_layouts():
    assert gemm_form("NN", BF16, 8, 4, 2048, 2048) == ("tiled", 256, 256)
    assert gemm_form("MT", BF16, 8, 4096, 2048, 2048) == ("tiled", 256, 256)
    assert gemm_form("MT", BF16, 8, 4096, 2048, 2048, gathered=True)[0] == "staged"
    assert gemm_form("MT", FP32, 8, 4096, 2048, 2048, gathered=True) == ("tiled", 128, 128)
