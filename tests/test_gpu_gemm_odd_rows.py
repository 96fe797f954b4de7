"""16-bit products on a B in rows that are no whole aligned 16-byte chunks, read as it is: edges of the tiles, every place of a row's
last chunk, a K that ends inside a step, one to four pairs of steps.  Which products take that kernel is asserted where no GPU is
needed."""

import multiprocessing

import pytest
import torch

from tests import recorded_launches as rec

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
# M, N, K, elements between the rows of B, elements in front of B
SIZES = [(1000, 4097, 1000, 0, 0), (100, 50257, 64, 0, 0), (1030, 5001, 8, 0, 0), (900, 8100, 72, 0, 0), (700, 6005, 128, 3, 1),
         (640, 7006, 136, 0, 0), (640, 7007, 192, 0, 3), (640, 5120, 200, 0, 1), (640, 5128, 256, 1, 0), (513, 8447, 264, 5, 7),
         (2048, 3999, 328, 0, 0), (128, 20008, 64, 4, 0), (1500, 3002, 512, 0, 5)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("M,N,K,pad,offset", SIZES)
def test_odd_rows(M, N, K, pad, offset, dtype):
    """Integer operands: the f32 sum is exact in any order, so every element has one right bit pattern.  B ends with its memory;
    between its rows is NaN."""
    from lighthouse_amd import ops

    g = torch.Generator(device="cuda").manual_seed(M + N)
    draw = lambda *shape: torch.randint(-3, 4, shape, device="cuda", generator=g).float()  # noqa: E731
    a, b, bias = draw(M, K), draw(K, N), draw(N)
    want = a @ b
    memory = torch.full((offset + (K - 1) * (N + pad) + N,), float("nan"), device="cuda", dtype=DTYPES[dtype])
    view = memory[offset:].as_strided((K, N), (N + pad, 1))
    view.copy_(b)
    a = a.to(DTYPES[dtype])
    assert torch.equal(ops.gemm(a, view, out_dtype=torch.float32), want)
    got = ops.gemm(a, view, bias.to(DTYPES[dtype]), relu=True)
    assert torch.equal(got, torch.relu(want + bias).to(DTYPES[dtype]))


def _names(so, sizes, f32=False):
    r = rec.Recorder(so)
    found = {}
    for M, N, K, pad, offset in sizes:
        for dt in (rec._lib.BF16, rec._lib.F16):
            rc, launches = r.calls("lh_hip_gemm", 1 << 50, 2 << 50, (3 << 50) + 2 * offset, 4 << 50, M, N, K, K, N + pad, N, dt,
                                   rec._lib.F32 if f32 else dt, 1, None)
            assert rc == 0, r.lib.lh_hip_last_error()
            found[M, N, K, pad, offset, dt] = [launch.name for launch in launches]
    return found


def test_who_takes_odd_rows(tmp_path):
    """The sizes above are one launch, with or without a step that K ends in; rows of whole aligned chunks, more than a round of
    workgroups, and a long K that is cut instead are other kernels'."""
    others = [(1000, 4096, 1000, 0, 0), (1000, 4096, 1000, 8, 8), (4096, 4097, 1024, 0, 0), (200, 2049, 8192, 0, 0), (1000, 4097, 1001, 0, 0)]
    with multiprocessing.get_context("spawn").Pool(1) as pool:
        found = pool.apply(_names, (rec.build(tmp_path), SIZES + others))
    for (M, N, K, pad, offset, dt), names in found.items():
        if (M, N, K, pad, offset) in others:
            assert not any("gemm16_odd_rows" in n for n in names), (M, N, K, names)
        else:
            assert len(names) == 1 and f"gemm16_odd_rowsILi{1 if dt == rec._lib.BF16 else 2}ELb{int(K % 64 != 0)}E" in names[0], (M, N, K, names)


def test_few_rows_stay_on_the_small_tiles(tmp_path):
    """Where they are the faster kernels, and for every f32 result that they take: their sums over eight shares of K are nearer to
    64 bits than one chain.  A long K with two workgroups on a CU is faster on a copy."""
    small = [(8, 14521, 1552, 0, 0), (32, 13636, 2344, 0, 0), (1, 15466, 792, 0, 0), (2319, 267, 368, 0, 0)]
    odd = [(256, 12202, 536, 0, 0), (196, 5130, 264, 0, 0), (2747, 442, 472, 0, 0)]  # (f32 results: the small tiles)
    both = [(3353, 541, 3528, 0, 0), (1000, 4097, 1000, 0, 0), (100, 50257, 768, 0, 0), (3146, 1547, 2560, 0, 0)]
    copied = [(3146, 1547, 2784, 0, 0), (4928, 903, 2944, 0, 0)]
    kind = lambda names: "small" if "gemm_small" in names[0] else "odd" if "gemm16_odd_rows" in names[0] else "copied"  # noqa: E731
    with multiprocessing.get_context("spawn").Pool(1) as pool:
        so = rec.build(tmp_path)
        for f32, expected in ((False, {"small": small, "odd": odd + both, "copied": copied}), (True, {"small": small + odd, "odd": both, "copied": copied})):
            for want, sizes in expected.items():
                for size, names in pool.apply(_names, (so, sizes, f32)).items():
                    assert kind(names) == want and (len(names) > 1) == (want == "copied"), (size, f32, names)
