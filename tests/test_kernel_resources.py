"""Registers of the built kernels, from the metadata their code objects carry (no GPU): what a change of one part of a kernel does
to the occupancy of all its workgroups shows here and hardly in a time."""

from __future__ import annotations

import struct

import msgpack


def _metadata(blob: bytes):
    """Every kernel's record in a shared object's bundles of gfx950 code objects."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = blob.find(magic)
    while at >= 0:
        (entries,), p = struct.unpack_from("<Q", blob, at + 24), at + 32
        for _ in range(entries):
            offset, size, length = struct.unpack_from("<QQQ", blob, p)
            triple, p = blob[p + 24:p + 24 + length], p + 24 + length
            if size and b"gfx950" in triple:
                yield from _notes(blob[at + offset:at + offset + size])
        at = blob.find(magic, at + 24)


def _notes(elf: bytes):
    (table,), (entry, count) = struct.unpack_from("<Q", elf, 0x28), struct.unpack_from("<HH", elf, 0x3A)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, table + i * entry + 4)
        p, size = struct.unpack_from("<QQ", elf, table + i * entry + 0x18)
        end = p + size
        while kind == 7 and p < end:  # SHT_NOTE
            name, length, note = struct.unpack_from("<III", elf, p)
            p += 12 + (name + 3) // 4 * 4
            if note == 32:  # NT_AMDGPU_METADATA
                yield from msgpack.unpackb(elf[p:p + length], strict_map_key=False)["amdhsa.kernels"]
            p += (length + 3) // 4 * 4


def _kernels():
    from torchllmtuner_amd import _lib

    with open(_lib.LIB_PATH, "rb") as f:
        return {k[".name"]: k for k in _metadata(f.read())}


def test_the_plans_second_launch_leaves_a_cu_its_places():
    """64 registers are eight waves a SIMD, all there are: the rare workgroups of this launch, of which a lane holds many loads, must not
    cost the others theirs."""
    found = {n: k for n, k in _kernels().items() if "route_rows_kernel" in n}
    assert len(found) == 4  # 512 and 1024 lanes, with and without statistics
    for name, k in found.items():
        assert k[".vgpr_count"] <= 64 and k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, name


def test_no_kernel_keeps_vector_registers_in_memory():
    spilled = {n: k[".vgpr_spill_count"] for n, k in _kernels().items() if k[".vgpr_spill_count"]}
    # (four registers of the gate's backward on matrix tiles)
    assert all("gate_bwd_kernel" in n and v <= 4 for n, v in spilled.items()), spilled
