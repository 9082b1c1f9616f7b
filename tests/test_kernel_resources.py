"""What the compiler gave the kernels of the built library, by the notes of its code objects."""
import struct

import msgpack
import pytest

from vllm_gguf_plugin_prism_amd import _lib

# Kernels whose registers are counted out: a value that goes to scratch is a trip through memory, per tile or per step.
# (IQ3_S with one tile of rows and two column groups: three registers, and faster than with one group by 3 %)
EXCEPT = ("6TIQ3_SELi1ELi2E",)
WHOLE_IN_REGISTERS = ("mmqf_kernel", "tile_stream_kernel", "tile_dealt_kernel", "tile_dealt_pair_kernel", "tile_wide_kernel", "tile_expert_kernel", "mmvq_pair_kernel")


def kernels(data: bytes):
    """(name, bytes of scratch per lane) of every kernel in the code objects bundled in a library."""
    bundle = data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while bundle >= 0:
        entry = bundle + 32
        for _ in range(struct.unpack_from("<Q", data, bundle + 24)[0]):
            at, size, length = struct.unpack_from("<QQQ", data, entry)
            if b"gfx950" in data[entry + 24:entry + 24 + length]:
                yield from _notes(data[bundle + at:bundle + at + size])
            entry += 24 + length
        bundle = data.find(b"__CLANG_OFFLOAD_BUNDLE__", bundle + 1)


def _notes(elf: bytes):
    sections, (entry_size, count) = struct.unpack_from("<Q", elf, 40)[0], struct.unpack_from("<HH", elf, 58)
    for i in range(count):
        _, kind, _, _, at = struct.unpack_from("<IIQQQ", elf, sections + i * entry_size)
        if kind != 7:                                        # SHT_NOTE
            continue
        name, size, note = struct.unpack_from("<III", elf, at)
        if note == 32:                                       # NT_AMDGPU_METADATA
            at += 12 + (name + 3) // 4 * 4
            for kernel in msgpack.unpackb(elf[at:at + size])["amdhsa.kernels"]:
                yield kernel[".name"], kernel[".private_segment_fixed_size"]


@pytest.fixture(scope="module")
def scratch():
    if not _lib.LIB_PATH.exists():
        from vllm_gguf_plugin_prism_amd import build
        build.build()
    return dict(kernels(_lib.LIB_PATH.read_bytes()))


@pytest.mark.parametrize("kernel", WHOLE_IN_REGISTERS)
def test_nothing_goes_to_scratch(kernel, scratch):
    of = {name: n for name, n in scratch.items() if f"{len(kernel)}{kernel}I" in name}   # (mangled: length, name, template arguments)
    assert of and not {name: n for name, n in of.items() if n and not any(e in name for e in EXCEPT)}


# the tile of the matrix instruction, a property of the format (measured: csrc/mmq_f_core.h)
@pytest.mark.parametrize("fmt,tile", [("5FQ4_K", 32), ("5FQ5_K", 32), ("5FQ6_K", 16)])
def test_tile_of_the_prefill_gemm(fmt, tile, scratch):
    of = [name for name in scratch if "11mmqf_kernelI" in name and fmt in name]
    assert of and all(f"Li{tile}E" in name for name in of)
