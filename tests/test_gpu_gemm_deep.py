"""The tiles of problems that give no CU a second workgroup: one to six stages of K and more than the rings hold, edges of the
tiles, a K that ends inside a step, both layouts of B, every kind of output."""

import multiprocessing
import re

import pytest
import torch

from tests import recorded_launches as rec

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


SIZES = [(2048, 2048, 64), (2048, 2048, 128), (2000, 2040, 192), (2048, 2048, 256), (1921, 1928, 320), (2048, 2048, 384),
         (1929, 2000, 72), (1930, 2000, 200), (1000, 4096, 1000), (1999, 1992, 264), (1537, 2304, 768),
         # more than a CU's worth of 128 x 128 tiles: 128 x 192, 256 x 128, 128 x 256
         (8192, 768, 320), (8192, 768, 448), (8191, 760, 384), (8129, 768, 640), (4090, 1528, 512), (4096, 1536, 1024),
         (4096, 2048, 512), (4096, 2048, 2048), (4096, 2000, 576), (4090, 2048, 768), (3900, 2000, 1000), (2048, 4096, 448), (2000, 4000, 1032), (1999, 4088, 640)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,transpose_b", [("bf16", False), ("bf16", True), ("f16", False), ("f16", True)])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_one_tile_per_cu(M, N, K, dtype, transpose_b):
    """Integer operands: the f32 sum is exact in any order, so every element has one right bit pattern."""
    from lighthouse_amd import ops

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    draw = lambda *shape: torch.randint(-2, 3, shape, device="cuda", generator=g).float()  # noqa: E731
    a, b, bias, c = draw(M, K), draw(K, N), draw(N), draw(M, N)
    want = a @ b
    dt = DTYPES[dtype]
    a, b = a.to(dt), (b.T.contiguous() if transpose_b else b).to(dt)
    assert torch.equal(ops.gemm(a, b, bias.to(dt), relu=True, transpose_b=transpose_b), torch.relu(want + bias).to(dt))
    out = torch.empty(M, N, device="cuda")
    assert torch.equal(ops.gemm(a, b, bias, out=out, residual=c, transpose_b=transpose_b), want + c + bias)
    out16 = torch.empty(M, N, device="cuda", dtype=dt)
    assert torch.equal(ops.gemm(a, b, out=out16, residual=c.to(dt), transpose_b=transpose_b), (want + c).to(dt))


def _tiles(so):
    r, found = rec.Recorder(so), set()
    for M, N, K in SIZES:
        for dt in (rec._lib.BF16, rec._lib.F16):
            for out in (dt, rec._lib.F32):
                for flags, ldb in ((0, N), (16, K)):
                    rc, launches = r.calls("lh_hip_gemm", 1 << 50, 2 << 50, 3 << 50, 4 << 50, M, N, K, K, ldb, N, dt, out, flags, None)
                    assert rc == 0, r.lib.lh_hip_last_error()
                    found |= {m.groups() for m in (re.search(r"gemm16_deepILi(\d)ELi(\d)ELi(\d)ELb(\d)ELb(\d)ELb(\d)E", n.name) for n in launches) if m}
    return {tuple(int(v) for v in f) for f in found}


def test_the_sizes_reach_every_tile(tmp_path):
    """Type; rows / 64; columns / 128 (3: 192); edges; K ends inside a step, which 192 columns do not take; B stored [N, K]."""
    with multiprocessing.get_context("spawn").Pool(1) as pool:
        found = pool.apply(_tiles, (rec.build(tmp_path),))
    for tile in ((2, 1), (2, 2), (4, 1)):
        assert {f[3:] for f in found if f[1:3] == tile} == {(e, t, b) for e, t in ((0, 0), (1, 0), (1, 1)) for b in (0, 1)}, tile
    assert {f[3:] for f in found if f[1:3] == (2, 3)} == {(e, 0, b) for e in (0, 1) for b in (0, 1)}
    assert {f[0] for f in found} == {rec._lib.BF16, rec._lib.F16}


# M, N, K, cuts (None: the library's choice): pieces of two, three, four, five and more stages of K, where the rings hold four
CUTS = [(128, 512, 256, 2), (100, 520, 384, 2), (129, 512, 768, 4), (256, 1000, 2048, 8), (200, 1000, 640, 2), (256, 512, 5120, 8), (300, 1000, 4096, None),
        (1000, 1000, 4096, None), (512, 768, 3072, None), (1024, 1024, 8192, None)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,transpose_b", [("bf16", False), ("bf16", True), ("f16", False), ("f16", True)])
@pytest.mark.parametrize("M,N,K,cuts", CUTS)
def test_cut_along_k(M, N, K, cuts, dtype, transpose_b):
    """Integer operands, as above."""
    from lighthouse_amd import ops

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    draw = lambda *shape: torch.randint(-2, 3, shape, device="cuda", generator=g).float()  # noqa: E731
    a, b, bias = draw(M, K), draw(K, N), draw(N)
    want = a @ b
    dt = DTYPES[dtype]
    a, b = a.to(dt), (b.T.contiguous() if transpose_b else b).to(dt)
    assert torch.equal(ops.gemm(a, b, out_dtype=torch.float32, transpose_b=transpose_b, split_k=cuts), want)
    assert torch.equal(ops.gemm(a, b, bias.to(dt), relu=True, transpose_b=transpose_b, split_k=cuts), torch.relu(want + bias).to(dt))


def _cuts(so):
    r, found = rec.Recorder(so), []
    requests = {None: 0, **{n: rec._lib.GEMM_SPLITK[n] for n in (2, 4, 8)}}
    for M, N, K, cuts in CUTS:
        for dt in (rec._lib.BF16, rec._lib.F16):
            for flags, ldb in ((0, N), (16, K)):
                rc, launches = r.calls("lh_hip_gemm", 1 << 50, 2 << 50, 3 << 50, 4 << 50, M, N, K, K, ldb, N, dt, dt, flags | requests[cuts], None)
                assert rc == 0 and len(launches) == 2, r.lib.lh_hip_last_error()
                m = re.search(r"gemm16_deepILi(\d)ELi2ELi1ELb(\d)ELb0ELb(\d)ELb1E", launches[0].name)
                assert m, (M, N, K, cuts, launches[0].name)
                g = launches[0].gemm
                assert launches[0].grid == -(-M // 128) * -(-N // 128) * g.splits <= 256 and g.splits * g.K == K and g.splits == (cuts or g.splits)
                found.append((dt, int(m.group(2)), int(m.group(3)), g.K // 64))
    return found


def test_the_cuts_reach_every_kernel(tmp_path):
    """Type, edges, B stored [N, K]: on pieces shorter than the rings, as long, and longer."""
    with multiprocessing.get_context("spawn").Pool(1) as pool:
        found = pool.apply(_cuts, (rec.build(tmp_path),))
    assert {p for *_, p in found} >= {2, 3, 4, 5}
    for kernel in {f[:3] for f in found}:
        stages = [f[3] for f in found if f[:3] == kernel]
        assert min(stages) < 4 < max(stages), kernel
    assert len({f[:3] for f in found}) == 8
