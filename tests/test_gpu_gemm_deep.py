"""The 128-row tiles of problems that give no CU a second workgroup: one to six stages of K and more than the rings hold, edges of the
tile, a K that ends inside a step, both layouts of B, every kind of output."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


@pytest.mark.parametrize("dtype,transpose_b", [("bf16", False), ("bf16", True), ("f16", False), ("f16", True)])
@pytest.mark.parametrize("M,N,K", [(2048, 2048, 64), (2048, 2048, 128), (2000, 2040, 192), (2048, 2048, 256), (1921, 1928, 320), (2048, 2048, 384),
                                   (2047, 2056, 72), (1930, 2000, 200), (1000, 4096, 1000), (1999, 1992, 264), (1537, 2304, 768),
                                   # 192 columns: an output of that many on more rows, whole and with edges
                                   (8192, 768, 64), (8192, 768, 448), (8191, 760, 192), (8129, 768, 128), (5461, 1144, 512)])
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
