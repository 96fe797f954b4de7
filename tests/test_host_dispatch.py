"""What the library's host code makes of a call, on any machine: which kernels it launches on which addresses, and what memory it
takes.  The calls run on a recorder in the place of the HIP runtime (hip_recorder.cpp), in a process of its own."""

import ctypes
import multiprocessing
import random
import re

import pytest

from tests import recorded_launches as rec

DT = rec._lib.BF16
OUT, A, B, BIAS, WORKSPACE = (1 << 50, 2 << 50, 3 << 50, 4 << 50, 5 << 50)  # far apart, aligned


@pytest.fixture(scope="module")
def recorded(tmp_path_factory):
    """recorded(check, *args): check(recorder, *args) in a process whose library launches nothing."""
    so = rec.build(tmp_path_factory.mktemp("recorder"))
    with multiprocessing.get_context("spawn").Pool(1) as pool:
        yield lambda check, *args: pool.apply(_on_recorder, (so, check, args))


_recorder = None


def _on_recorder(so, check, args):
    global _recorder
    _recorder = _recorder or rec.Recorder(so)
    return check(_recorder, *args)


def _product(rng, largest):
    """A 16-bit product: any layout, row stride, alignment, K and output type."""
    size = lambda lo, hi: int(lo * (hi / lo) ** rng.random())  # noqa: E731
    while True:
        M, N, K = size(1, 8192), size(1, 8192), size(1, 8192)
        if rng.random() < 0.7:
            K = max(K // 8 * 8, 8)
        if rng.random() < 0.5:
            N = max(N // 8 * 8, 8)
        if 2 * M * N * K <= largest:
            break
    ta, tb = rng.random() < 0.3, rng.random() < 0.4
    stride = lambda cols: rng.choice([cols, cols, (cols + 63) // 64 * 64, cols + 8, cols + 1, (cols + 127) // 128 * 128 + 64])  # noqa: E731
    offset = lambda: 2 * rng.choice([0, 0, 1, 4, 8])  # noqa: E731
    return dict(M=M, N=N, K=K, lda=stride(M if ta else K), ldb=stride(K if tb else N), ldc=stride(N), a=A + offset(), b=B + offset(),
                out_dtype=rng.choice([DT, rec._lib.F32]), flags=(8 if ta else 0) | (16 if tb else 0) | rng.choice([0, 0, 1, 3, 33, 4]))


def _shape(p):
    return [p[k] for k in ("M", "N", "K", "lda", "ldb", "ldc")] + [DT, p["out_dtype"], p["flags"]]


def _pointers(p):
    return OUT, p["a"], p["b"], BIAS


def _row(M, N, K, lda=None, ldb=None, offset_a=0, offset_b=0, flags=0):
    return dict(M=M, N=N, K=K, lda=lda or (M if flags & 8 else K), ldb=ldb or (K if flags & 16 else N), ldc=N, a=A + 2 * offset_a,
                b=B + 2 * offset_b, out_dtype=DT, flags=flags)


# A off 16 bytes in rows that start on 128-byte lines: on a copy its rows do not, and the K that the kernels want is another.
COPIED_A = [_row(4096, 8192, 1000, lda=1024, offset_a=1), _row(2064, 5480, 1224, lda=1280, offset_a=1),
            _row(2560, 5120, 3000, lda=3072, offset_a=1), _row(8192, 3072, 760, lda=768, offset_a=1),
            _row(4096, 8192, 1000, lda=1024, offset_a=1, flags=16), _row(4096, 8192, 1001, lda=1024),
            # ... and a transposed B that would be copied into more than 32-bit offsets reach
            _row(300, 1100000, 1000, lda=1000, offset_a=1, flags=16)]


def _copies_once(r):
    rng = random.Random(7)
    problems = COPIED_A + [_product(rng, 2 * 8192 * 8192 * 2048) for _ in range(4000)]
    for p in problems:
        for _ in range(2):  # (the pool's buffers grow in the first call)
            rc, launches = r.calls("lh_hip_gemm", *_pointers(p), *_shape(p), None)
            assert rc == 0, (p, r.lib.lh_hip_last_error())
            written = []
            for launch in launches:
                copies = launch.copies
                for _, (lo, hi) in copies:
                    assert not any(lo < end and begin < hi for begin, end in written), f"a copy of a copy: {p}"
                written += [dst for dst, _ in copies]


def test_an_operand_is_copied_once(recorded):
    """A copy of a copy is wasted, and in the library's own memory it may be the same buffer."""
    recorded(_copies_once)


# A transposed A of fewer rows than the small-tile kernels take; B transposed off 16 bytes; K inside a step.
FEW_ROWS = [_row(M, 64, 1000, flags=8) for M in range(1, 8)] + [_row(4, 64, 1000, offset_b=1, flags=24), _row(1, 768, 3208, flags=8),
                                                              _row(64, 8, 4, offset_b=1, flags=16)]


def _queried_memory(r):
    rng = random.Random(11)
    problems = COPIED_A + FEW_ROWS + [_product(rng, rng.choice([2 << 22, 2 * 8192 * 8192 * 512])) for _ in range(8000)]
    for p in problems:
        need = r.lib.lh_hip_gemm_workspace_bytes_for(*_pointers(p), *_shape(p))
        rc, launches = r.calls("lh_hip_gemm_ws", *_pointers(p), *_shape(p), WORKSPACE if need else None, need, None)
        assert rc == 0, (p, need, r.lib.lh_hip_last_error())
        for launch in launches:
            for (lo, hi), _ in launch.copies:
                assert WORKSPACE <= lo and hi <= WORKSPACE + need, p


def test_a_workspace_of_the_queried_size_is_enough(recorded):
    recorded(_queried_memory)


def _offsets(r):
    """Products whose B, with K up to the end of the last step, lies on either side of 2^30 elements."""
    in_place = set()  # (the K's whose B was read where it is, on the near side of the limit)
    for K in (8, 40, 72, 96, 104, 200, 328, 1000, 4104):
        steps = (K + 63) // 64 * 64
        strides = {n + d for n in ((1 << 30) // steps // 8 * 8, (1 << 30) // K // 8 * 8, (1 << 29) // K // 8 * 8) for d in (-8, 0, 8)}
        for ldb in sorted(strides):
            for N in (520, ldb):
                rc, launches = r.calls("lh_hip_gemm", OUT, A, B, BIAS, 512, N, K, K, ldb, N, DT, DT, 0, None)
                assert rc == 0, r.lib.lh_hip_last_error()
                for launch in launches:
                    if "gemm16_direct" not in launch.name:
                        continue
                    g = launch.gemm
                    assert (g.K + 63) // 64 * 64 * g.ldb < 1 << 30, (K, N, ldb)
                    if "tail" in launch.name and launch.gemm.ldb == ldb:
                        in_place.add(K)
    assert in_place >= {200, 328, 1000}


def test_offsets_of_the_last_step_fit_32_bits(recorded):
    """The loads of a step that K ends in are addressed up to the end of the step, also those that touch no memory."""
    recorded(_offsets)


def _kernel(r, *args):
    rc, launches = r.calls(*args, None)
    assert rc == 0 and len(launches) == 1, r.lib.lh_hip_last_error()
    return launches[0].name


def _large_results(r):
    f32 = rec._lib.F32
    past_the_caches = lambda ldc, M=4096, N=4096, out=DT: _kernel(  # noqa: E731
        r, "lh_hip_gemm", OUT, A, B, BIAS, M, N, 4096, 4096, N, ldc, DT, out, 0).endswith("ELb1EEEvNS_8GemmArgsE")
    assert past_the_caches(50432, 8192, 50432) and past_the_caches(8192, 8192, 8192, f32)
    assert not past_the_caches(4096) and not past_the_caches(65536) and not past_the_caches(65536, out=f32)
    fp8 = lambda ldc, N: _kernel(r, "lh_hip_gemm_fp8", OUT, A, B, 1.0, 1.0, 8192, N, 8192, 8192, N, ldc, DT)  # noqa: E731
    assert "gemm8_directILb0ELb1E" in fp8(8192, 8192)
    assert "gemm8_directILb0ELb0E" in fp8(65536, 4096)


def test_columns_of_a_wide_buffer_are_no_large_result(recorded):
    """What counts is what is written, not the rows that it lies in."""
    recorded(_large_results)


def _touching(r):
    def touches(M, N, K, flags=0):
        rc, launches = r.calls("lh_hip_gemm", OUT, A, B, BIAS, M, N, K, K, K if flags & 16 else N, N, DT, DT, flags, None)
        assert rc == 0 and len(launches) == 1 and "gemm16_direct" in launches[0].name, r.lib.lh_hip_last_error()
        return bool(launches[0].gemm.touch_b)

    for flags in (0, 16):  # (1152 tiles of 128 x 128 on 512 workgroups, 288 on as many)
        assert [touches(8192, 2304, K, flags) for K in (128, 448, 512, 768, 1792, 2048)] == [False, False, True, True, True, False]
        assert [touches(3072, 1536, K, flags) for K in (448, 504, 512, 520)] == [False, False, True, True]


def test_a_long_enough_b_of_few_lines_is_touched(recorded):
    """What the direct kernels touch at the start: from K = 512 on, up to 128 lines of B for every workgroup."""
    recorded(_touching)


def _normed(r, sizes):
    """The tiles (rows, columns of 16) and widths (of 128) of the launches that normalise rows and multiply them, by size and type."""
    lib, found = rec._lib, {}
    for T, C in sizes:
        for dtype, separate in ((lib.BF16, False), (lib.F16, True)):
            p = lib.NanoGPTBlockParams()
            for i, (name, _) in enumerate(p._fields_):
                missing = ("w_qkv", "b_qkv") if separate else ("w_q", "w_k", "w_v")
                setattr(p, name, None if name in missing else B + (i << 32))
            opts = lib.NanoGPTBlockOpts(0 if separate else 1, lib.ACT_RELU if separate else lib.ACT_GELU_TANH,
                                        lib.F32 if separate else dtype, 4 * C)
            need = r.lib.lh_hip_nanogpt_block_workspace_bytes(1, T, C, dtype, ctypes.byref(opts))
            rc, launches = r.calls("lh_hip_nanogpt_block", OUT, A, ctypes.byref(p), 1, T, C, C // 64, 1e-5, dtype, ctypes.byref(opts),
                                   WORKSPACE, need, None)
            assert rc == 0, r.lib.lh_hip_last_error()
            kernels = [re.search(r"gemm_normed_kernelILi\dELi(\d)ELi(\d)ELi8ELi(\d)E", launch.name) for launch in launches]
            found[T, C, dtype] = [tuple(int(v) for v in k.groups()) for k in kernels if k]
    return found


def test_sizes_of_normed_products(recorded):
    """The sizes that the one launch is tested at take it: every width on every tile, bf16 with one weight matrix and f16 with
    three, and the widths that are no multiple of 128 do not."""
    from tests.test_gpu_block_normed import SIZES

    found = recorded(_normed, SIZES)
    for (T, C, dtype), kernels in found.items():
        assert bool(kernels) == (C % 128 == 0), (T, C)
        assert all(width == C // 128 for _, _, width in kernels)
    for dtype in (rec._lib.BF16, rec._lib.F16):
        reached = {k for (_, _, d), kernels in found.items() if d == dtype for k in kernels}
        assert reached == {(*tile, width) for tile in ((1, 2), (1, 4), (2, 4)) for width in range(1, 9)}


def _copies_that_pay(r):
    def launches(M, N, K, offset_b=0):
        p = _row(M, N, K, offset_b=offset_b, flags=8)
        rc, found = r.calls("lh_hip_gemm", *_pointers(p), *_shape(p), None)
        assert rc == 0, r.lib.lh_hip_last_error()
        return len(found)

    for M, N in ((1, 64), (4, 512), (7, 4096)):
        assert [launches(M, N, K) for K in (8, 24, 72, 80, 136)] == [1, 1, 1, 2, 2]
        assert [launches(M, N, K, 1) for K in (8, 24, 72, 136)] == [1, 1, 1, 1]
        assert launches(M, 64, 520, 1) == 2
    # ... on a caller's memory where there is room
    p = _row(4, 512, 1000, flags=8)
    for room, expected in ((0, 1), (7936, 1), (8192, 2), (1 << 20, 2)):
        rc, found = r.calls("lh_hip_gemm_ws", *_pointers(p), *_shape(p), WORKSPACE, room, None)
        assert rc == 0 and len(found) == expected, (room, r.lib.lh_hip_last_error())


def test_a_few_rows_are_untransposed_where_that_pays(recorded):
    """Fewer rows of a transposed A than the small-tile kernels take, K inside a step: a copy and the tile kernels, or one launch."""
    recorded(_copies_that_pay)
