"""Registers and scratch of the built kernels, from the notes of their code objects: what a kernel must not take, where taking it costs
half its waves or sends its operands through memory."""
import struct

import pytest

msgpack = pytest.importorskip("msgpack")


def _code_objects(data: bytes):
    """The gfx950 code objects of every source's bundle in the library."""
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := data.find(magic, at)) >= 0:
        here = at + len(magic)
        count, = struct.unpack_from("<Q", data, here)
        here += 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, here)
            target = data[here + 24:here + 24 + length]
            here += 24 + length
            if target.endswith(b"gfx950"):
                yield data[at + offset:at + offset + size]
        at += len(magic)


def _notes(elf: bytes):
    """The kernels' entries of a code object's note section."""
    sections, = struct.unpack_from("<Q", elf, 0x28)
    size, count = struct.unpack_from("<HH", elf, 0x3a)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, sections + i * size + 4)
        if kind != 7:                                    # SHT_NOTE
            continue
        offset, = struct.unpack_from("<Q", elf, sections + i * size + 0x18)
        name, length, kind = struct.unpack_from("<III", elf, offset)
        if kind == 32:                                   # NT_AMDGPU_METADATA
            start = offset + 12 + (name + 3) // 4 * 4
            yield from msgpack.unpackb(elf[start:start + length], raw=False)["amdhsa.kernels"]


@pytest.fixture(scope="module")
def kernels():
    from leone_amd.csrc import build
    with open(build.build(force=False), "rb") as handle:
        data = handle.read()
    found = {k[".name"]: k for elf in _code_objects(data) for k in _notes(elf)}
    assert len(found) > 500
    return found


def test_products_that_carry_out_a_norm(kernels):
    """Four waves a SIMD (128 registers of 512) and nothing in scratch."""
    normed = [k for name, k in kernels.items() if "gemm_fused_kernelILi1E" in name]
    assert len(normed) >= 40
    for k in normed:
        assert k[".vgpr_count"] <= 128 and k[".private_segment_fixed_size"] == 0, k[".name"]


def test_layer_norms_of_few_rows(kernels):
    """What takes rows element by element has a thread an element of every 1,024: five waves a SIMD, nothing in scratch."""
    normed = {name: k for name, k in kernels.items() if "add_layernorm_" in name}
    assert not [name for name, k in normed.items() if k[".private_segment_fixed_size"]]
    single = [k for name, k in normed.items() if "add_layernorm_single" in name]
    assert len(single) == 8 and all(k[".vgpr_count"] <= 96 and k[".max_flat_workgroup_size"] == 1024 for k in single)


def test_norms_behind_a_sublayer_of_short_rows(kernels):
    """Rows of up to 1,024 elements take a run a thread: eight waves a SIMD, or seven with eight places on their way."""
    held = [k for name, k in kernels.items() if "add_normed_held_kernel" in name and "Li1ELi" in name]
    assert sorted(k[".vgpr_count"] <= 64 for k in held) == [False, False, True, True] and all(k[".vgpr_count"] <= 72 for k in held)


def test_rms_norms_in_registers(kernels):
    """Rows of up to 4,096 elements keep four waves a SIMD, rows of up to 8,192 two, whatever the types."""
    for chunks, most in ((4, 128), (8, 256)):
        normed = [k for name, k in kernels.items() if "add_rmsnorm_vec_kernel" in name and f"Li256ELi{chunks}E" in name]
        assert len(normed) == 8
        for k in normed:
            assert k[".vgpr_count"] <= most and k[".private_segment_fixed_size"] == 0, k[".name"]


def test_gated_products_of_many_rows(kernels):
    """Six tiles of rows a wave, and four under a row-major weight, leave three waves a SIMD (168 registers of 512) where one wave takes
    a tile of the weight."""
    gated = [k for name, k in kernels.items() if "gemm_rows_kernelILi6ELi4ELi1ELi2ELi1ELi2E" in name
             or ("gemm_rows_kernelILi4ELi4ELi1ELi4ELi1ELi2E" in name and "Lb0EEE" in name)]
    assert len(gated) == 3 and all(k[".vgpr_count"] <= 168 for k in gated)


def test_float_products(kernels):
    """Nothing in scratch; where the weights are streamed, four waves a SIMD (their loads are what counts), in tiles three."""
    streams = [k for name, k in kernels.items() if "gemm_f32_few_kernel" in name or "gemm_f32_stream_kernel" in name]
    tiles = [k for name, k in kernels.items() if "gemm_f32_tile_kernel" in name]
    assert len(streams) == 16 and len(tiles) == 8
    for k, most in [(k, 128) for k in streams] + [(k, 168) for k in tiles]:
        assert k[".vgpr_count"] <= most and k[".private_segment_fixed_size"] == 0, k[".name"]


def test_attention_with_mixed_scores(kernels):
    """What 32 heads of 128 leave to scratch, with keys of their own and with keys that four share, and no more; smaller ones less or nothing."""
    found = {name.split("attention_talk_prefill_kernel")[1][:24]: k[".private_segment_fixed_size"] for name, k in kernels.items()
             if "attention_talk_prefill_kernel" in name}
    assert len(found) == 16 and found.pop("ILi128ELi32ELi4ELi1EEEvN") <= 100 and found.pop("ILi128ELi32ELi4ELi4EEEvN") <= 176
    assert max(found.values()) <= 80 and not any(size for name, size in found.items() if name.startswith("ILi64E"))
