"""The small-tile GEMM kernels: tile and K edges, every layout, unaligned views, each element type."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32, "fp8": torch.float8_e4m3fn}


def _matrix(rows, cols, dtype, seed, pad):
    """Integers -3 .. 3 as a column range of a wider matrix whose other columns hold NaN: a kernel that counts
    anything outside the operand shows it."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    v = torch.randint(-3, 4, (rows, cols), device="cuda", generator=g).float()
    buf = torch.full((rows, cols + 2 * pad), float("nan"), device="cuda").to(DTYPES[dtype])
    buf[:, pad:pad + cols] = v.to(DTYPES[dtype])
    return buf[:, pad:pad + cols], v


@pytest.mark.parametrize("pad", [0, 1])
@pytest.mark.parametrize("dtype,layout", [(d, l) for d in ("bf16", "f16", "f32") for l in ("nn", "nt", "tn", "tt")] + [("fp8", "nn")])
@pytest.mark.parametrize("shape", [(16, 16, 16),       # one tile, less than a k-step of 16-bit values
                                   (17, 65, 64),       # one past a tile in both directions
                                   (33, 31, 63),       # K one short of a step
                                   (100, 129, 65),     # ... and one past it
                                   (1, 1000, 513), (250, 33, 1100), (64, 2050, 97),
                                   (300, 300, 777)])   # the larger tiles
def test_small_tiles(shape, dtype, layout, pad):
    """Integer operands: the f32 sum is exact in any order, so the result has one right bit pattern."""
    from lighthouse_amd import ops

    M, N, K = shape
    ta, tb = layout[0] == "t", layout[1] == "t"
    a, av = _matrix(K if ta else M, M if ta else K, dtype, 1, pad)
    b, bv = _matrix(N if tb else K, K if tb else N, dtype, 2, pad)
    want = (av.T if ta else av).double() @ (bv.T if tb else bv).double()
    out = torch.full((M, N + 2), 7.0, device="cuda")
    view = out[:, :N]
    if dtype == "fp8":
        ops.gemm_fp8(a, b, 0.5, 2.0, out=view)
        assert torch.equal(view.double(), want)
    else:
        bias = torch.arange(N, device="cuda").float() % 5 - 2
        ops.gemm(a, b, bias, out=view, relu=True, transpose_a=ta, transpose_b=tb)
        assert torch.equal(view.double(), torch.relu(want + bias.double()))
        ops.gemm(a, b, out=view, accumulate_c=True, transpose_a=ta, transpose_b=tb)
        assert torch.equal(view.double(), torch.relu(want + bias.double()) + want)
        if dtype != "f32":  # 16-bit output: one rounding of the exact sum
            got = ops.gemm(a, b, transpose_a=ta, transpose_b=tb)
            assert torch.equal(got, want.to(DTYPES[dtype]))
    assert bool((out[:, N:] == 7.0).all())


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("shape,offset", [((2100, 2051, 64), 0),    # N odd: 128- and 256-wide tiles that end inside a row
                                          ((2304, 2304, 128), 1),   # whole tiles, rows that start 2 (4) bytes off
                                          ((600, 8190, 96), 3)])
def test_tile_kernels_write_any_alignment(shape, offset, dtype):
    """Problems too large for the small tiles whose result, bias and accumulator input are not 16-byte aligned:
    the tile kernels write them in place, and nothing beside them."""
    from lighthouse_amd import ops

    M, N, K = shape
    a, av = _matrix(M, K, dtype, 3, 0)
    b, bv = _matrix(K, N, dtype, 4, 0)
    want = av.double() @ bv.double()
    for out_dtype in {DTYPES[dtype], torch.float32}:
        buf = torch.full((M, N + 5), 7.0, device="cuda", dtype=out_dtype)
        view = buf[:, offset:offset + N]
        bias = (torch.arange(N + 1, device="cuda").float() % 5 - 2).to(out_dtype)[1:]
        ops.gemm(a, b, bias, out=view)
        assert torch.equal(view, (want + bias.double()).to(out_dtype))
        view.copy_(view.clamp(-8, 8).round())
        before = view.double().clone()
        ops.gemm(a, b, out=view, accumulate_c=True)
        assert torch.equal(view, (want + before).to(out_dtype))
        assert bool((buf[:, :offset] == 7.0).all()) and bool((buf[:, offset + N:] == 7.0).all())


@pytest.mark.parametrize("dtype,M,N,K", [("bf16", 457, 5401, 901), ("f16", 457, 5401, 901), ("f32", 345, 5237, 166)])
def test_a_problem_copied_for_the_tile_kernels_runs_on_them(dtype, M, N, K):
    """Here the tile kernels plus padded copies of both operands beat the small tiles on the operands as they are, by
    little: once the copies are made the tile kernels run.  They add up k in one order whatever the tile, the
    small tiles in another, so the f32 sums have the bits of the same product on operands that need no copy."""
    from lighthouse_amd import ops

    g = torch.Generator(device="cuda").manual_seed(7)
    a = torch.randn(M, K, device="cuda", generator=g).to(DTYPES[dtype])
    b = torch.randn(K, N, device="cuda", generator=g).to(DTYPES[dtype])
    a0, b0 = torch.zeros(M, (K + 63) // 64 * 64, device="cuda", dtype=a.dtype), torch.zeros((K + 63) // 64 * 64, N + 7, device="cuda", dtype=a.dtype)
    a0[:, :K], b0[:K, :N] = a, b
    want = ops.gemm(a0, b0, out_dtype=torch.float32)[:, :N]
    assert torch.equal(ops.gemm(a, b, out_dtype=torch.float32), want)


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_rows_that_split_dwords_are_priced(dtype):
    """k-contiguous operands whose rows start at odd elements go through the L1 at a fraction of the rate: this product runs
    on copies for the tile kernels (same bits as a requested tile on aligned operands), not on the small tiles."""
    from lighthouse_amd import ops

    M, N, K = 1408, 1024, 2368
    g = torch.Generator(device="cuda").manual_seed(8)
    a, b = (torch.randn(rows, K, device="cuda", generator=g).to(DTYPES[dtype]) for rows in (M, N))
    odd_a, odd_b = torch.empty(M, K + 1, device="cuda", dtype=a.dtype)[:, 1:], torch.empty(N, K + 1, device="cuda", dtype=a.dtype)[:, 1:]
    odd_a.copy_(a), odd_b.copy_(b)
    want = ops.gemm(a, b, transpose_b=True, out_dtype=torch.float32, tile=(128, 128))
    assert torch.equal(ops.gemm(odd_a, odd_b, transpose_b=True, out_dtype=torch.float32), want)


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_a_second_round_of_small_tiles_is_priced(dtype):
    """1.3 workgroups of small tiles per compute unit take nearly as long as 2: cut along K the tile kernel is faster."""
    from lighthouse_amd import ops

    g = torch.Generator(device="cuda").manual_seed(9)
    a = torch.randn(672, 3072, device="cuda", generator=g).to(DTYPES[dtype])
    b = torch.randn(3072, 512, device="cuda", generator=g).to(DTYPES[dtype])
    want = ops.gemm(a, b, out_dtype=torch.float32, split_k=4)
    assert torch.equal(ops.gemm(a, b, out_dtype=torch.float32), want)


def test_fp8_operand_copies_are_priced_as_they_are_made():
    """One launch copies both operands of an fp8 product into aligned rows: faster here than the small tiles on codes whose
    rows start at odd addresses.  The sums have the bits of the same product on aligned codes."""
    from lighthouse_amd import ops

    M, N, K = 752, 4984, 2176
    g = torch.Generator(device="cuda").manual_seed(10)
    a = torch.randn(M, K, device="cuda", generator=g).to(torch.float8_e4m3fn)
    b = torch.zeros(K, N + 8, device="cuda", dtype=torch.float8_e4m3fn)
    b[:, :N] = torch.randn(K, N, device="cuda", generator=g).to(torch.float8_e4m3fn)
    odd_a = torch.empty(M, K + 1, device="cuda", dtype=a.dtype)[:, 1:]
    odd_a.copy_(a)
    want = ops.gemm_fp8(a, b, 0.5, 2.0, out_dtype=torch.float32)[:, :N]
    assert torch.equal(ops.gemm_fp8(odd_a, b[:, :N].contiguous(), 0.5, 2.0, out_dtype=torch.float32), want)


def test_only_the_operands_that_are_copied_are_priced():
    """A few rows of an odd stride next to an aligned B: copying the rows costs little, and the product cut along K is faster than
    small tiles on rows that split dwords.  The sums have the bits of the requested cut on aligned operands."""
    from lighthouse_amd import ops

    g = torch.Generator(device="cuda").manual_seed(11)
    a = torch.randn(16, 6144, device="cuda", generator=g).to(torch.bfloat16)
    b = torch.randn(6144, 2048, device="cuda", generator=g).to(torch.bfloat16)
    odd = torch.empty(16, 6145, device="cuda", dtype=a.dtype)[:, 1:]
    odd.copy_(a)
    want = ops.gemm(a, b, out_dtype=torch.float32, split_k=8)
    assert torch.equal(ops.gemm(odd, b, out_dtype=torch.float32), want)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("dtype", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("shape,offset", [((2100, 2051, 64), 0), ((2304, 2304, 128), 1),
                                          ((2100, 2050, 4096), 3)])  # a long K
def test_tile_kernels_write_any_alignment_in_every_layout(shape, offset, dtype, layout):
    """Transposed operands too, with bias and activation, on exactly the workspace that the query gives."""
    from lighthouse_amd import ops

    M, N, K = shape
    ta, tb = layout[0] == "t", layout[1] == "t"
    a, av = _matrix(M, K, dtype, 5, 0)
    b, bv = _matrix(K, N, dtype, 6, 0)
    a, b = (a.T.contiguous() if ta else a), (b.T.contiguous() if tb else b)
    want = av.double() @ bv.double()
    for out_dtype in {DTYPES[dtype], torch.float32}:
        buf = torch.full((M, N + 5), 7.0, device="cuda", dtype=out_dtype)
        view = buf[:, offset:offset + N]
        bias = (torch.arange(N + 1, device="cuda").float() % 5 - 2).to(out_dtype)[1:]
        options = {"transpose_a": ta, "transpose_b": tb}
        need = ops.gemm_workspace_bytes(M, N, K, DTYPES[dtype], out_dtype, bias=True, relu=True, operands=(view, a, b, bias), **options)
        workspace = torch.empty((need + 255) // 256 * 256, dtype=torch.uint8, device="cuda")
        ops.gemm(a, b, bias, out=view, relu=True, workspace=workspace, **options)
        assert torch.equal(view, torch.relu(want + bias.double()).to(out_dtype))
        ops.gemm(a, b, bias, out=view, gelu=True, **options)  # the bits of the same product into aligned rows
        wide = torch.empty((M, (N + 7) // 8 * 8), device="cuda", dtype=out_dtype)[:, :N]
        assert torch.equal(view, ops.gemm(a, b, bias, out=wide, gelu=True, **options))
        assert bool((buf[:, :offset] == 7.0).all()) and bool((buf[:, offset + N:] == 7.0).all())
