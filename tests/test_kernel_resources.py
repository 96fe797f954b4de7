"""What the compiler gave the kernels of the built library: registers where a launch counts on two workgroups per compute
unit.  Read from the metadata notes of the library's own code objects."""

import re
import struct
import subprocess

import pytest

from lighthouse_amd import _lib

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled name: {metadata key: value}} of every kernel in the library."""
    _lib.load()
    blob = _lib.library_path().read_bytes()
    obj = tmp_path_factory.mktemp("code") / "object"
    found, at = {}, blob.find(MAGIC)
    while at >= 0:
        pos = at + len(MAGIC) + 8
        for _ in range(struct.unpack_from("<Q", blob, pos - 8)[0]):
            offset, size, length = struct.unpack_from("<QQQ", blob, pos)
            target, pos = blob[pos + 24:pos + 24 + length], pos + 24 + length
            if size and b"gfx950" in target:
                obj.write_bytes(blob[at + offset:at + offset + size])
                notes = subprocess.run([READELF, "--notes", str(obj)], capture_output=True, text=True, check=True).stdout
                for kernel in re.split(r"\n +- \.agpr_count", notes)[1:]:
                    name = re.search(r"\.name: +(\S+)", kernel).group(1)
                    found[name] = {k: int(v) for k, v in re.findall(r"\.(\w+): +(\d+)", kernel)}
        at = blob.find(MAGIC, at + 1)
    assert len(found) > 100
    return found


def test_two_128x128_gemm_workgroups_fit_a_compute_unit(kernels):
    """Eight waves each: two workgroups are four waves per SIMD, which have 128 registers each."""
    tiles = {n: k["vgpr_count"] for n, k in kernels.items() if re.search(r"gemm16_directILi[12]ELi2ELi1E", n)}
    assert len(tiles) == 16  # bf16 / f16, whole / edge tiles, whole / cut K, B [K, N] / [N, K]
    assert {n: v for n, v in tiles.items() if v > 128} == {}


def test_only_wide_element_access_attention_uses_scratch(kernels):
    """A kernel that touches scratch memory at all costs microseconds more per dispatch.  The attention kernels that load
    element by element at the widths 224 (f32) and 256 are the ones that do."""
    scratch = {n for n, k in kernels.items() if k["private_segment_fixed_size"] > 0}
    assert {n for n in scratch if not re.search(r"attention16_anyd_kernelILi[12]ELi8ELi2E|attention32_anyd_kernelILi[78]ELi2E", n)} == set()


def test_small_tile_gemms_are_built_for_the_layouts_that_exist(kernels):
    """Six tiles; four layouts of a 16-bit or f32 product, one of an fp8 product, whose operands are never transposed."""
    small = [re.search(r"gemm_small_kernelILi(\d)E", n) for n in kernels]
    of_type = [int(m.group(1)) for m in small if m]
    assert {t: of_type.count(t) for t in set(of_type)} == {_lib.F32: 24, _lib.BF16: 24, _lib.F16: 24, _lib.F8E4M3: 6}
