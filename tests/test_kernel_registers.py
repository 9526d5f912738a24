"""Registers of the built kernels, from the metadata of their code objects."""
import os
import struct

import pytest

msgpack = pytest.importorskip("msgpack")

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ramses_amd", "libramses_hip.so")


def _notes(elf):
    """The AMDGPU metadata note (type 32) of an ELF64 image."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    shentsize, shnum = struct.unpack_from("<HH", elf, 58)
    for i in range(shnum):
        kind, = struct.unpack_from("<I", elf, shoff + i * shentsize + 4)
        if kind != 7:  # SHT_NOTE
            continue
        at, size = struct.unpack_from("<QQ", elf, shoff + i * shentsize + 24)
        end = at + size
        while at < end:
            namesz, descsz, ntype = struct.unpack_from("<III", elf, at)
            desc = at + 12 + (namesz + 3) // 4 * 4
            if ntype == 32:
                yield msgpack.unpackb(elf[desc:desc + descsz])
            at = desc + (descsz + 3) // 4 * 4


def _kernels():
    data = open(LIB, "rb").read()
    magic, out, at = b"__CLANG_OFFLOAD_BUNDLE__", {}, 0
    while (at := data.find(magic, at)) >= 0:
        count, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(count):
            offset, size, idlen = struct.unpack_from("<QQQ", data, p)
            if b"amdgcn" in data[p + 24:p + 24 + idlen] and size:
                for note in _notes(data[at + offset:at + offset + size]):
                    out.update({k[".name"]: k for k in note["amdhsa.kernels"]})
            p += 24 + idlen
        at += 1
    return out


def test_staged_sweep_does_not_spill():
    """The oct-tree's staged solve with 7-point slopes and a solver fixed at
    compile time (amr_unsplit<double, solver, false, slope>): its registers
    hold it."""
    if not os.path.exists(LIB):
        pytest.skip("the library is not built")
    staged = {n: k for n, k in _kernels().items() if "amr_unsplitIdLi" in n and "ELb0E" in n and "Li99E" not in n}
    assert len(staged) == 6, sorted(staged)
    for n, k in staged.items():
        assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, n
