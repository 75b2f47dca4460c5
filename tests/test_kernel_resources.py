"""What the compiler gave the attention kernels over codes (pitch_attn_codes.hip), read from the code object metadata
that the built library carries: no kernel has scratch memory or spilled registers. Scratch shows in no result, but its
loads and stores stand in a tile's loop and make it wait for every load in flight."""
import struct

import pytest

from pitch_amd import _lib

BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data: bytes):
    """The device code objects of the library's offload bundles."""
    at = data.find(BUNDLE)
    while at >= 0:
        entries, = struct.unpack_from("<Q", data, at + len(BUNDLE))
        p = at + len(BUNDLE) + 8
        for _ in range(entries):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            if b"amdgcn" in data[p + 24:p + 24 + length]:
                yield data[at + offset:at + offset + size]
            p += 24 + length
        at = data.find(BUNDLE, p)


def _kernels(elf: bytes):
    """The kernels of a code object's metadata note (AMDGPU, type 32)."""
    import msgpack
    table, = struct.unpack_from("<Q", elf, 40)
    entry, count = struct.unpack_from("<HH", elf, 58)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, table + i * entry + 4)
        offset, size = struct.unpack_from("<QQ", elf, table + i * entry + 24)
        if kind != 7 or size == 0:   # SHT_NOTE
            continue
        name, length, note = struct.unpack_from("<III", elf, offset)
        if note == 32:
            start = offset + 12 + (name + 3) // 4 * 4
            yield from msgpack.unpackb(elf[start:start + length])["amdhsa.kernels"]


def test_attention_over_codes_uses_no_scratch():
    pytest.importorskip("msgpack")
    if not _lib.LIB_PATH.exists():
        pytest.skip("HIP library not built")
    found = [k for elf in _code_objects(_lib.LIB_PATH.read_bytes()) for k in _kernels(elf)
             if "attn_codes" in k[".name"]]
    assert len(found) == 2 * 6 * 9 * 2    # dimensions, kinds of caches, widths of keys and values, four or eight heads
    for k in found:
        used = [k[".private_segment_fixed_size"], k[".vgpr_spill_count"], k[".sgpr_spill_count"]]
        assert used == [0, 0, 0], (k[".name"], used)
