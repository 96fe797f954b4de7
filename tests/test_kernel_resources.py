"""What the compiler made of the kernels of the built library: registers where a launch counts on two workgroups per compute
unit, scratch memory, loads.  Read from the library's own code objects, their metadata notes and their instructions."""

import re
import struct
import subprocess

import pytest

from lighthouse_amd import _lib

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled name: {metadata key: value, "object": path of its code object}} of every kernel in the library."""
    _lib.load()
    blob = _lib.library_path().read_bytes()
    folder = tmp_path_factory.mktemp("code")
    found, at = {}, blob.find(MAGIC)
    while at >= 0:
        pos = at + len(MAGIC) + 8
        for _ in range(struct.unpack_from("<Q", blob, pos - 8)[0]):
            offset, size, length = struct.unpack_from("<QQQ", blob, pos)
            target, pos = blob[pos + 24:pos + 24 + length], pos + 24 + length
            if size and b"gfx950" in target:
                obj = folder / f"object{at + offset}"
                obj.write_bytes(blob[at + offset:at + offset + size])
                notes = subprocess.run([READELF, "--notes", str(obj)], capture_output=True, text=True, check=True).stdout
                for kernel in re.split(r"\n +- \.agpr_count", notes)[1:]:
                    name = re.search(r"\.name: +(\S+)", kernel).group(1)
                    found[name] = {k: int(v) for k, v in re.findall(r"\.(\w+): +(\d+)", kernel)}
                    found[name]["object"] = obj
        at = blob.find(MAGIC, at + 1)
    assert len(found) > 100
    return found


def test_two_128x128_gemm_workgroups_fit_a_compute_unit(kernels):
    """Eight waves each: two workgroups are four waves per SIMD, which have 128 registers each."""
    tiles = {n: k["vgpr_count"] for n, k in kernels.items() if re.search(r"gemm16_direct(_tail)?ILi[12]ELi2ELi1E", n)}
    # bf16 / f16, B [K, N] / [N, K]: whole / edge tiles by whole / cut K, and a K that ends inside a step
    assert len(tiles) == 16 + 4 and sum("tail" in n for n in tiles) == 4
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


def test_what_to_touch_is_an_argument_of_the_touching_kernels_alone(kernels):
    """Arguments cost every dispatch of a kernel, whether a call of it touches the weights of later launches or not."""
    touching = {n for n in kernels if "5Touch" in n}
    assert touching and all(re.search(r"gemm_small_touchingILi\dE", n) for n in touching)
    assert not any(f"touchingILi{_lib.F8E4M3}E" in n for n in touching)
    for n in touching:  # (each has a twin that takes none)
        twin = n.replace("NS_5TouchE", "").replace("19gemm_small_touching", "17gemm_small_kernel").replace("EEEvNS_8Gemm", "ELb1ELb0EEEvNS_8Gemm")
        assert kernels[twin]["kernarg_segment_size"] + 40 == kernels[n]["kernarg_segment_size"], n


def test_cut_gemms_load_without_loops_over_resources(kernels):
    """The panels of a workgroup are the same for its lanes: a load whose resource the compiler holds in vector registers sits
    in a loop over the lanes' resources (exec is narrowed right before it), which the kernels cut along K once had in
    their main loop."""
    cut = {n: k["object"] for n, k in kernels.items() if re.search(r"gemm16_directILi[12]ELi2ELi1ELb[01]ELb1E", n)}
    assert len(cut) == 8
    for obj in set(cut.values()):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(obj)], capture_output=True, text=True, check=True).stdout
        assert "buffer_load_dwordx4" in text and " lds" in text
        assert not re.search(r"s_and_saveexec_b64[^\n]*\n(?:\s+s_nop[^\n]*\n)*\s+buffer_load_dwordx4[^\n]* lds", text)
