"""What the compiler notes about the built kernels: those whose registers are their limit keep them out of scratch memory."""
import re
import struct

import pytest

from butterfly_amd import ops

msgpack = pytest.importorskip("msgpack")


def _notes(elf):
    """The metadata notes (type 32) of one code object."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    size, count = struct.unpack_from("<HH", elf, 58)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, shoff + i * size + 4)
        at, length = struct.unpack_from("<QQ", elf, shoff + i * size + 24)
        end = at + length
        while kind == 7 and at < end:                  # SHT_NOTE
            name, desc, type_ = struct.unpack_from("<III", elf, at)
            at += 12 + (name + 3) // 4 * 4
            if type_ == 32:
                yield msgpack.unpackb(elf[at:at + desc])
            at += (desc + 3) // 4 * 4


def _spilled():
    """Vector registers spilled, by mangled kernel name."""
    with open(ops.library_path(), "rb") as f:
        lib = f.read()
    out = {}
    for bundle in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", lib):
        at = bundle.end()
        entries, = struct.unpack_from("<Q", lib, at)
        at += 8
        for _ in range(entries):
            off, size, name = struct.unpack_from("<QQQ", lib, at)
            target = lib[at + 24:at + 24 + name]
            at += 24 + name
            if b"gfx950" in target and size:
                for note in _notes(lib[bundle.start() + off:bundle.start() + off + size]):
                    out.update((k[".name"], k[".vgpr_spill_count"]) for k in note["amdhsa.kernels"])
    return out


@pytest.mark.parametrize("kernel", ["attn_window_mfma_kernelILi2ELi16E", "attn_window_mfma_kernelILi4ELi8E", "attn_decode_flat_kernel", "gemm_big4_kernel"])
def test_kernels_without_spills(kernel):
    if not ops.load_library():
        pytest.skip("kernel library not built")
    found = {n: s for n, s in _spilled().items() if kernel in n}
    assert found and not any(found.values()), found
