"""f32 results of the tile GEMM kernels in rows that do not start at multiples of 64 bytes, launches whose workgroups start
late, and a K that ends inside a step of 64."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


@pytest.mark.parametrize("dtype,transpose_b", [("bf16", False), ("bf16", True), ("f16", False)])
@pytest.mark.parametrize("M,N,K,pad,offset", [(129, 9001, 64, 0, 0),      # 128 x 128 tiles, the last of 41 columns
                                              (300, 16641, 64, 0, 0),     # ... and of one column, fewer than stand in front of a piece
                                              (2050, 3000, 128, 4, 0),    # rows 16 bytes past a piece, each by 16 more
                                              (1024, 8192, 64, 1, 3),     # whole tiles, every phase of a row
                                              (513, 8197, 192, 8, 7),
                                              (4096, 9216, 64, 5, 1),     # several rounds of the large tiles
                                              (4100, 8450, 64, 0, 0)])
def test_rows_between_pieces(M, N, K, pad, offset, dtype, transpose_b):
    """Integer operands: the f32 sum is exact in any order, so every element has one right bit pattern."""
    from lighthouse_amd import ops

    g = torch.Generator().manual_seed(M + N)
    draw = lambda *shape: torch.randint(-3, 4, shape, generator=g).float()
    a, b, bias = draw(M, K), draw(N, K) if transpose_b else draw(K, N), draw(N)
    want = (a @ (b.T if transpose_b else b)).cuda()
    a, b = a.cuda().to(DTYPES[dtype]), b.cuda().to(DTYPES[dtype])
    buf = torch.full((offset + M * (N + pad),), 7.0, device="cuda")
    rows = buf[offset:].view(M, N + pad)
    out = rows[:, :N]
    for extra in ({}, {"relu": True}):
        want_now = torch.relu(want + bias.cuda()) if extra else want
        out.fill_(float("nan"))
        ops.gemm(a, b, bias.cuda() if extra else None, out=out, transpose_b=transpose_b, **extra)
        assert torch.equal(out, want_now)
        assert bool((rows[:, N:] == 7.0).all()) and bool((buf[:offset] == 7.0).all())


@pytest.mark.parametrize("M,N", [(2048, 33280),    # 1040 tiles of 256 x 256: four rounds and 16 tiles, half the workgroups start late
                                 (2048, 45056),    # 5.5 rounds: those that have a tile fewer do
                                 (2048, 65536)])   # eight whole rounds: half of them do
def test_workgroups_that_start_late(M, N):
    from lighthouse_amd import ops

    g = torch.Generator(device="cuda").manual_seed(N)
    a, b = (torch.randint(-3, 4, s, device="cuda", generator=g).float() for s in ((M, 64), (64, N)))
    got = ops.gemm(a.bfloat16(), b.bfloat16())
    assert torch.equal(got, (a @ b).bfloat16())


@pytest.mark.parametrize("dtype,layout", [("bf16", "nn"), ("bf16", "nt"), ("f16", "tn")])
@pytest.mark.parametrize("M,N,K", [(1000, 4096, 1000),   # 128 x 128 tiles, the step ends after 40 of 64
                                   (1030, 4104, 72),     # one chunk of the second step
                                   (900, 8200, 8),       # less than a step
                                   (700, 5000, 120), (2048, 8192, 328), (2100, 6152, 184), (640, 12288, 568),
                                   (100, 40000, 104)])
def test_k_that_ends_inside_a_step(M, N, K, dtype, layout):
    """Operands whose rows go on behind K, with NaN: what the last step reads past K must count as nothing."""
    from lighthouse_amd import ops

    g = torch.Generator(device="cuda").manual_seed(M * K)
    ta, tb = layout[0] == "t", layout[1] == "t"
    av, bv = (torch.randint(-3, 4, s, device="cuda", generator=g).float() for s in ((M, K), (K, N)))

    def stored(v, transposed):
        v = v.T if transposed else v
        buf = torch.full((v.shape[0] + 72, v.shape[1] + 72), float("nan"), device="cuda").to(DTYPES[dtype])
        buf[:v.shape[0], :v.shape[1]] = v.to(DTYPES[dtype])
        return buf[:v.shape[0], :v.shape[1]]

    a, b = stored(av, ta), stored(bv, tb)
    want = av @ bv
    got = ops.gemm(a, b, out_dtype=torch.float32, transpose_a=ta, transpose_b=tb)
    assert torch.equal(got, want)
    bias = torch.randint(-3, 4, (N,), device="cuda", generator=g).to(DTYPES[dtype])
    got = ops.gemm(a, b, bias, relu=True, transpose_a=ta, transpose_b=tb)
    assert torch.equal(got, torch.relu(want + bias.float()).to(DTYPES[dtype]))


@pytest.mark.parametrize("dtype,transpose_b", [("bf16", False), ("f16", True)])
@pytest.mark.parametrize("M,N,K,lda", [(4096, 8192, 1000, 1024), (2064, 5480, 1224, 1280), (2100, 6152, 72, 128)])
def test_rows_off_16_bytes_and_a_k_inside_a_step(M, N, K, lda, dtype, transpose_b):
    """A is copied for its alignment.  Its own rows start on 128-byte lines and the copy's do not, which the choice of what K is
    padded to depends on; one copy is made all the same, in the library's memory (the second call finds its buffers
    large enough) and in a workspace of the queried size."""
    from lighthouse_amd import ops

    g = torch.Generator(device="cuda").manual_seed(M * K)
    av, bv = (torch.randint(-3, 4, s, device="cuda", generator=g).float() for s in ((M, K), (K, N)))
    buf = torch.full((M, lda), float("nan"), device="cuda").to(DTYPES[dtype])
    a = buf[:, 1:1 + K]
    a.copy_(av)
    b = (bv.T if transpose_b else bv).contiguous().to(DTYPES[dtype])
    want = av @ bv
    for _ in range(2):
        assert torch.equal(ops.gemm(a, b, out_dtype=torch.float32, transpose_b=transpose_b), want)
    out = torch.empty((M, N), device="cuda")
    need = ops.gemm_workspace_bytes(M, N, K, DTYPES[dtype], torch.float32, transpose_b=transpose_b, operands=(out, a, b, None))
    ops.gemm(a, b, out=out, transpose_b=transpose_b, workspace=torch.empty(need, dtype=torch.uint8, device="cuda"))
    assert torch.equal(out, want)


@pytest.mark.parametrize("M,N,K,offset_b", [(1, 64, 1000, 0), (4, 64, 1000, 0), (7, 512, 1048, 0), (4, 64, 1000, 1)])
def test_few_rows_of_a_transposed_a_on_a_workspace(M, N, K, offset_b):
    """Small products whose K ends inside a step need no memory of a caller's: the queried size is 0, and enough.  They take it
    where there is room for their copies."""
    from lighthouse_amd import ops

    g = torch.Generator(device="cuda").manual_seed(M + K)
    a, bv = (torch.randint(-3, 4, s, device="cuda", generator=g).bfloat16() for s in ((K, M), (K, N)))
    b = torch.zeros(offset_b + N * K, device="cuda", dtype=torch.bfloat16)[offset_b:].view((N, K) if offset_b else (K, N))
    b.copy_(bv.T if offset_b else bv)
    out = torch.empty((M, N), device="cuda")
    options = {"transpose_a": True, "transpose_b": bool(offset_b)}
    need = ops.gemm_workspace_bytes(M, N, K, torch.bfloat16, torch.float32, operands=(out, a, b, None), **options)
    assert need == 0
    want = a.float().T @ bv.float()
    for size in (need, 1 << 20):
        ops.gemm(a, b, out=out.fill_(float("nan")), workspace=torch.empty(size, dtype=torch.uint8, device="cuda"), **options)
        assert torch.equal(out, want)
    assert torch.equal(ops.gemm(a, b, out_dtype=torch.float32, **options), want)
