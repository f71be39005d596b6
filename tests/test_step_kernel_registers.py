"""Registers of the default step kernels as built: they decide how many
wavefronts a SIMD holds (512 registers a lane in blocks of 8), and packed beds
of some 100k particles and more are slower by several percent with one fewer.
Read from the metadata the compiler writes beside each kernel."""
import os
import struct

import msgpack
import pytest

LIB = os.path.join(os.path.dirname(__file__), "..", "liggghts-public_amd", "libdem_amd.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _device_elfs(blob):
    at = blob.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", blob, at + 24)
        p = at + 32
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", blob, p)
            name = blob[p + 24:p + 24 + length]
            p += 24 + length
            if b"gfx950" in name:
                yield blob[at + offset:at + offset + size]
        at = blob.find(MAGIC, at + 24)


def _kernels():
    with open(LIB, "rb") as f:
        blob = f.read()
    out = {}
    for elf in _device_elfs(blob):
        phoff, = struct.unpack_from("<Q", elf, 32)
        phsize, phnum = struct.unpack_from("<HH", elf, 54)
        for k in range(phnum):
            kind, _, offset = struct.unpack_from("<IIQ", elf, phoff + k * phsize)
            if kind != 4:  # PT_NOTE
                continue
            nname, ndesc, _ = struct.unpack_from("<III", elf, offset)
            desc = offset + 12 + (nname + 3) // 4 * 4
            meta = msgpack.unpackb(elf[desc:desc + ndesc])
            out.update({q[".name"]: q for q in meta["amdhsa.kernels"]})
    return out


def _name(real, mesh, general):
    return f"_ZN3dem6k_stepI{real}Lb{mesh}ELi256ELi4ELb{general}ELi0ELi1EEEvNS_8StepArgsE"


@pytest.mark.parametrize("real,mesh,general,waves", [
    ("f", 0, 0, 4), ("f", 0, 1, 4), ("f", 1, 0, 4), ("f", 1, 1, 3),
    ("d", 0, 0, 3), ("d", 0, 1, 2), ("d", 1, 0, 3), ("d", 1, 1, 2)])
def test_wavefronts_of_the_default_step_kernel(real, mesh, general, waves):
    q = _kernels()[_name(real, mesh, general)]
    assert 512 // ((q[".vgpr_count"] + 7) // 8 * 8) >= waves
    assert q[".vgpr_spill_count"] == 0
