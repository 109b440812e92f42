"""The small tiles (32, 64, 128 and 192 rows of 128 columns) of the 16-bit tiled kernel: which calls take them, and every
layout and epilogue at the edges of their heights against float64 products."""

import ctypes

import pytest
import torch

from flash_model_architectures_amd import _native, ops
from oracle import torch_oracle as to

from .helpers import GEMM_ELEM_TOL, TOL, assert_close


KINDS = {"TN": 0, "NN": 1, "MT": 2}


def gemm_tile(kind: str, dtype, experts: int, rows: int, n: int, k: int, epilogue: int = 0) -> tuple:
    """(rows, columns) of the tallest tile of a call with contiguous, aligned operands."""

    args = _native.GroupedGemmArgs()
    args.struct_size = ctypes.sizeof(args)
    args.kind, args.dtype, args.epilogue = KINDS[kind], _native.DTYPE_CODE[dtype], epilogue
    args.num_experts, args.rows, args.n, args.k = experts, rows, n, k
    args.a = args.b = args.c = ctypes.c_void_p(1 << 20)
    out = [ctypes.c_int32() for _ in range(2)]
    assert _native.load().xma_grouped_gemm_tile(ctypes.byref(args), *(ctypes.byref(v) for v in out)) == 0
    return tuple(v.value for v in out)


@pytest.mark.parametrize(
    "kind,experts,rows,n,k,epilogue,tile",
    [
        # the benchmark's layers: many rows per expert and several rounds of tiles
        ("TN", 8, 16384, 28672, 4096, 1, (256, 256)),
        ("NN", 8, 16384, 14336, 4096, 2, (256, 256)),
        ("TN", 64, 98304, 2048, 1024, 0, (256, 256)),
        ("NN", 64, 98304, 2048, 2048, 0, (256, 256)),
        # experts' last rows, or too few tiles
        ("TN", 128, 12248, 1536, 2048, 1, (192, 128)),
        ("NN", 128, 12248, 2048, 1536, 0, (192, 128)),
        ("TN", 64, 18000, 2048, 2048, 1, (192, 128)),
        ("NN", 64, 9000, 2048, 2048, 0, (256, 256)),  # 118-121 us either way
        ("TN", 6, 12004, 512, 1024, 0, (128, 128)),
        ("NN", 6, 12004, 512, 1024, 0, (128, 128)),
        ("TN", 8, 400, 4096, 14336, 0, (192, 128)),
        ("NN", 8, 0, 4096, 4096, 0, (192, 128)),
        # weight gradients: two rounds of tiles, 330 rows per expert
        ("MT", 8, 16384, 4096, 14336, 0, (256, 256)),
        ("MT", 8, 2640, 2048, 2048, 0, (256, 256)),
        ("MT", 8, 2639, 2048, 2048, 0, (128, 128)),
        ("MT", 8, 16384, 2048, 1792, 0, (256, 256)),  # 100 us, 110 in small tiles
    ],
)
def test_which_calls_take_them(kind, experts, rows, n, k, epilogue, tile):
    for dtype in (torch.bfloat16, torch.float16):
        assert gemm_tile(kind, dtype, experts, rows, n, k, epilogue) == tile


@pytest.mark.parametrize(
    "experts,rows,n,k,large",
    [
        # long reductions in one round of large tiles, and in the greater part of a second one
        (8, 16000, 2048, 1024, True),
        (16, 8000, 1024, 1024, True),
        (8, 4000, 2048, 1792, True),
        (4, 16000, 4096, 1792, True),
        (2, 8000, 4096, 3584, True),
        (16, 500, 1024, 1024, False),
        # half a round, a quarter of a second one, and row tiles that leave XCDs without work
        (1, 9000, 2048, 1024, False),
        (6, 2000, 2048, 1408, False),
        (4, 4000, 768, 3072, False),
        # two rounds and more: the reduction's length, earlier the longer the launch
        (64, 281, 2048, 1024, False),
        (64, 400, 2048, 1024, True),
        (128, 230, 1024, 4096, False),
        (128, 300, 1024, 4096, True),
        (256, 180, 3584, 4096, True),
    ],
)
def test_tile_of_a_weight_gradient(experts, rows, n, k, large):
    """Against the times of both tiles (rows: of each expert)."""

    want = (256, 256) if large else (128, 128)
    assert gemm_tile("MT", torch.bfloat16, experts, experts * rows, n, k) == want


@pytest.mark.parametrize(
    "kind,experts,rows,n,k,epilogue,tile",
    [
        # experts' rows a little below and above a multiple of 192, of which small tiles need a second round
        ("TN", 4, 187, 28672, 4096, 1, (256, 256)),  # 231 us in 256 x 256, 362 in 192 x 128, 306 in 128 x 128
        ("NN", 4, 187, 14336, 4096, 2, (256, 256)),  # 119, 185, 162
        ("TN", 32, 187, 1536, 2048, 1, (256, 256)),  # 51, 74, 53
        ("TN", 8, 200, 6144, 2048, 0, (256, 256)),  # 48, 74, 54
        ("NN", 64, 200, 768, 2048, 2, (256, 256)),  # 64, 79, 66
        ("NN", 128, 160, 512, 2048, 0, (256, 256)),  # 72, 93, 91
        ("NN", 32, 187, 1792, 4096, 2, (256, 256)),  # 123, 178, 166
        ("TN", 16, 4000, 768, 3072, 0, (256, 256)),  # 236, 288, 316
        # rows that start in the middle of a line of 128 bytes
        ("TN", 32, 200, 520, 7528, 0, (256, 256)),  # 140, 235, 191
        ("TN", 64, 200, 15056, 520, 1, (256, 256)),  # 559, 731, 678
        ("NN", 128, 1000, 7528, 520, 2, (256, 256)),  # 2557, 2956, 2918
        # where they pay
        ("TN", 64, 281, 2048, 2048, 1, (192, 128)),  # 228, 205, 244
        ("TN", 16, 125, 1024, 4096, 0, (192, 128)),  # 61, 40, 43
        ("TN", 1, 9000, 1024, 512, 0, (192, 128)),  # 19, 14, 18
        ("NN", 6, 2000, 512, 1024, 2, (128, 128)),  # 41, 38, 34
    ],
)
def test_tile_of_a_projection(kind, experts, rows, n, k, epilogue, tile):
    """Against the times of the three tiles, in the comments (rows: of each expert)."""

    assert gemm_tile(kind, torch.bfloat16, experts, experts * rows, n, k, epilogue) == tile


def test_tile_of_the_other_kernels():
    assert gemm_tile("TN", torch.bfloat16, 128, 16, 1536, 2048) == (16, 32)
    assert gemm_tile("NN", torch.float32, 8, 1000, 256, 256)[1] == 128


# rows per expert: both sides of every height, a full tile and a last one of each height behind it, none
SIZES = [192, 193, 1, 31, 32, 33, 0, 64, 65, 128, 129, 200, 320, 321, 385, 95, 97, 191, 2, 0, 1, 0]
# (reduction, columns, tile of TN and of NN): one stage, a last stage of eight, whole ones, a partial last tile of columns; the
# gated epilogues need columns in multiples of 16: halves of 8, 72, 136 and 168, in tiles of 64 and 128
SMALL = [(8, 8, 192, 192), (72, 136, 192, 192), (320, 264, 192, 192), (456, 328, 192, 192)]
GATED = [(8, 16, 192, 192), (72, 144, 192, 192), (320, 272, 192, 192), (456, 336, 192, 192)]


def _setup(sizes, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    ends = torch.tensor(sizes).cumsum(0).tolist()
    offsets = torch.tensor([0] + ends, dtype=torch.int32, device="cuda")
    rows = [slice(end - size, end) for end, size in zip(ends, sizes)]
    index = torch.randperm(ends[-1], generator=g, device="cuda").int()
    return g, offsets, rows, index


def _products(rows, a, w):  # w[e]: [in, out]
    return torch.cat([a[r].double() @ w[e].double() for e, r in enumerate(rows)])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sizes", [SIZES, [3, 700]])
@pytest.mark.parametrize("k,n,tn,nn", SMALL + GATED)
def test_heights(k, n, tn, nn, sizes, dtype):
    E, M = len(sizes), sum(sizes)
    g, offsets, rows, index = _setup(sizes, k + n)
    if sizes is SIZES:
        assert gemm_tile("TN", dtype, E, M, n, k) == (tn, 128) and gemm_tile("NN", dtype, E, M, n, k) == (nn, 128)
    assert gemm_tile("MT", dtype, E, M, n, k) == (128, 128)

    def rand(*shape, scale=1.0):
        return (torch.randn(*shape, generator=g, device="cuda") * scale).to(dtype)

    def empty(*shape):
        return torch.full(shape, float("nan"), dtype=dtype, device="cuda")

    tol, elem = TOL[dtype], GEMM_ELEM_TOL[dtype]
    x, w, bias = rand(M, k), rand(E, n, k, scale=0.1), rand(E, n)
    gathered = x[index.long()]
    want = _products(rows, gathered, w.transpose(1, 2)).float()
    with_bias = want + torch.cat([bias[e].float().expand(r.stop - r.start, n) for e, r in enumerate(rows)])

    # TN: gathered rows in, grouped out; grouped in, scattered out, with a bias
    out = empty(M, n)
    ops.scatter2scatter(x, w.permute(0, 2, 1), index, index, out, 1, False, True, offsets)
    assert_close(out, want, tol, "TN", elem_tol=elem)
    out = empty(M, n)
    ops.scatter2scatter(gathered, w.permute(0, 2, 1), index, index, out, 1, True, False, offsets, bias)
    assert_close(out[index.long()], with_bias, tol, "TN, scattered", elem_tol=elem)

    # the activations' epilogues, gated ones over the halves of the columns
    for activation in ("swiglu", "glu", "gelu_tanh"):
        gated = activation != "gelu_tanh"
        if gated and (k, n, tn, nn) not in GATED:
            continue
        if gated and sizes is SIZES:
            epilogue, _, _ = ops.FUSED_ACTIVATIONS[activation]
            assert gemm_tile("TN", dtype, E, M, n, k, epilogue) == (tn, 128)
            assert gemm_tile("NN", dtype, E, M, n // 2, k, epilogue + 1) == (nn, 128)
        act, pre = empty(M, n // 2 if gated else n), empty(M, n)
        ops.up_projection_fused(x, w, index, offsets, act, pre, 1, activation, bias)
        assert_close(pre, with_bias, tol, f"{activation}, pre-activation", elem_tol=elem)
        module = {"swiglu": to.swiglu_packed, "glu": torch.nn.GLU(), "gelu_tanh": torch.nn.GELU(approximate="tanh")}[activation]
        assert_close(act, module(pre.float()), tol, activation)
        act2 = empty(*act.shape)
        ops.up_projection_fused(x, w, index, offsets, act2, None, 1, activation, bias)
        assert torch.equal(act, act2)

        # NN through the activation's backward; the product is rounded before it
        dy, w_down = rand(M, k), rand(E, k, act.size(1), scale=0.1)
        d_act = _products(rows, dy, w_down).to(dtype).float()
        leaf = pre.float().requires_grad_()
        module(leaf).backward(d_act)
        d_pre = empty(M, n)
        ops.down_projection_dgrad_fused(dy, w_down, pre, offsets, d_pre, activation)
        assert_close(d_pre, leaf.grad, tol, f"{activation} backward")

    # NN, scattered and grouped
    dy, w_nn = rand(M, k), rand(E, k, n, scale=0.1)
    want = _products(rows, dy, w_nn).float()
    for grouped in (True, False):
        out = empty(M, n)
        ops.scatter2scatter(dy, w_nn, index, index, out, 1, True, grouped, offsets)
        assert_close(out if grouped else out[index.long()], want, tol, "NN", elem_tol=elem)

    # MT: experts without rows get zeros
    dw = empty(E, n, k)
    dn = rand(M, n)
    ops.group_bwd_W(dn, gathered, offsets, dw.permute(0, 2, 1), E)
    want = torch.stack([dn[r].double().T @ gathered[r].double() for r in rows]).float()
    assert_close(dw, want, tol, "MT", elem_tol=elem)


@pytest.mark.gpu
@pytest.mark.parametrize("K", [4160, 6200, 8320])
@pytest.mark.parametrize("kind", ["TN", "NN"])
def test_split_reductions_of_every_height(kind, K):
    """Few tiles and long reductions: tiles of every height are cut in 2, 3 and 4 parts.  Small integers, whose sums are
    exact in any order: bit for bit."""

    sizes, N, dt = [200, 70, 130, 40, 10], 136, torch.bfloat16
    E, M = len(sizes), sum(sizes)
    g, offsets, rows, index = _setup(sizes, K)
    assert gemm_tile(kind, dt, E, M, N, K)[1] == 128
    for _ in range(2):
        a = torch.randint(-2, 3, (M, K), generator=g, device="cuda").to(dt)
        w = torch.randint(-1, 2, (E, K, N), generator=g, device="cuda").to(dt)
        want = _products(rows, a, w).to(dt)
        out = torch.full((M, N), float("nan"), dtype=dt, device="cuda")
        stored = w.transpose(1, 2).contiguous().permute(0, 2, 1) if kind == "TN" else w
        ops.scatter2scatter(a, stored, index, index, out, 1, True, True, offsets)
        assert torch.equal(out, want)


@pytest.mark.gpu
@pytest.mark.parametrize(
    "sizes,N", [([11200, 129, 128, 127, 257, 384, 385, 1, 0, 10240] * 2, 4104), ([2048, 2049, 4096, 2200], 8200)]
)
def test_flat_tiles_of_the_input_gradient(sizes, N):
    """256 columns: an expert's last rows in tiles of 128, and the halves of the tiles of a last round (124 and 106 tiles).
    Small integers, bit for bit."""

    dt, K = torch.bfloat16, 2056
    E, M = len(sizes), sum(sizes)
    assert gemm_tile("NN", dt, E, M, N, K) == gemm_tile("NN", dt, E, M, N, K, 2) == (256, 256)
    g, offsets, rows, index = _setup(sizes, M)
    a = torch.randint(-2, 3, (M, K), generator=g, device="cuda").to(dt)
    w = torch.randint(-1, 2, (E, K, N), generator=g, device="cuda").to(dt)
    want = _products(rows, a, w)
    out = torch.full((M, N), float("nan"), dtype=dt, device="cuda")
    ops.scatter2scatter(a, w, index, index, out, 1, True, False, offsets)
    assert torch.equal(out[index.long()], want.to(dt))
    saved = torch.randn(M, 2 * N, generator=g, device="cuda").to(dt)
    d_pre = torch.full((M, 2 * N), float("nan"), dtype=dt, device="cuda")
    ops.down_projection_dgrad_fused(a, w, saved, offsets, d_pre, "swiglu")
    leaf = saved.float().requires_grad_()
    to.swiglu_packed(leaf).backward(want.to(dt).float())
    assert_close(d_pre, leaf.grad, TOL[dt], "swiglu backward in flat tiles")


@pytest.mark.gpu
def test_table_of_tiles():
    """More experts than the kernel looks up itself: the tiles come from a table."""

    sizes = ([70, 0, 130, 5, 200] * 104)[:517]
    E, M, K, N = len(sizes), sum(sizes), 72, 136
    g, offsets, rows, index = _setup(sizes, 0)
    assert gemm_tile("TN", torch.bfloat16, E, M, N, K)[1] == 128
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = torch.randn(E, N, K, generator=g, device="cuda").bfloat16()
    out = torch.full((M, N), float("nan"), dtype=x.dtype, device="cuda")
    ops.scatter2scatter(x, w.permute(0, 2, 1), index, index, out, 1, True, True, offsets)
    assert_close(out, _products(rows, x, w.transpose(1, 2)).float(), TOL[x.dtype], "table", elem_tol=GEMM_ELEM_TOL[x.dtype])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize(
    "experts,columns", [(3, 8), (3, 520), (8, 8192), (8, 8200), (5, 333), (256, 36), (8, 16384), (9, 333), (12, 3333)]
)
def test_column_sums(experts, columns, dtype):
    """Per-expert column sums in blocks of every width, with vectors and without."""

    g = torch.Generator("cuda").manual_seed(columns)
    sizes = torch.randint(0, 700, (experts,), generator=g, device="cuda")
    sizes[0], sizes[1] = 0, 1
    offsets = torch.cat([sizes.new_zeros(1), sizes.cumsum(0)]).int()
    x = torch.randn(int(offsets[-1]), columns, generator=g, device="cuda").to(dtype)
    out = torch.full((experts, columns), float("nan"), dtype=dtype, device="cuda")
    ops.expert_colsum(x, offsets, out)
    ends = offsets.tolist()
    want = torch.stack([x[a:b].double().sum(0) for a, b in zip(ends, ends[1:])])
    # one rounding of the result, and the roundings of up to 700 additions in fp32, whose terms are about one
    rounding = torch.finfo(dtype).eps / 2
    assert bool(((out.double() - want).abs() <= rounding * 1.01 * want.abs() + 700 * 2.0**-24 * 30).all())
