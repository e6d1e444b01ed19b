"""The verify attention kernels keep their state in registers: no kernel of the
built library has scratch memory (spilled vector registers would be reloaded
inside the tile loops, each reload waiting for every copy in flight).  Read from
the code objects' metadata, no GPU."""
import struct

import pytest

import d2sd

msgpack = pytest.importorskip("msgpack")


def _code_objects(data):
    """gfx950 ELF images of the offload bundles in a library."""
    at = data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            off, size, n = struct.unpack_from("<QQQ", data, entry)
            if b"gfx950" in data[entry + 24:entry + 24 + n] and size:
                yield data[at + off:at + off + size]
            entry += 24 + n
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)


def _kernels(elf):
    """Entries of amdhsa.kernels (the AMDGPU metadata note, type 32) of a code object."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        _, kind, _, _, off, size = struct.unpack_from("<IIQQQQ", elf, shoff + i * shentsize)
        end = off + size
        while kind == 7 and off < end:  # SHT_NOTE
            name, desc, note = struct.unpack_from("<III", elf, off)
            at = off + 12 + (name + 3) // 4 * 4
            if note == 32:
                yield from msgpack.unpackb(elf[at:at + desc])["amdhsa.kernels"]
            off = at + (desc + 3) // 4 * 4


def test_verify_attention_kernels_use_no_scratch():
    with open(d2sd.LIB_PATH, "rb") as f:
        kernels = [k for elf in _code_objects(f.read()) for k in _kernels(elf) if "verify_attn_kernel" in k[".name"]]
    assert len(kernels) == 68
    # (a spill without scratch went to accumulation registers, scratch without a spill is not touched)
    spilled = {k[".name"]: (k[".private_segment_fixed_size"], k[".vgpr_spill_count"]) for k in kernels
               if k[".private_segment_fixed_size"] and k[".vgpr_spill_count"]}
    assert not spilled, f"scratch bytes per lane, spilled registers: {spilled}"
