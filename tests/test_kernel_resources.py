"""Registers of the force kernels, from the built library's code objects: none
keeps its operands in scratch memory (an order whose accumulators and source row
outgrow the registers runs several times slower and still gives right results,
so no other test shows it)."""
import struct

import msgpack
import pytest

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(data):
    """The gfx950 code objects of every offload bundle in a host library."""
    at = data.find(MAGIC)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(count):
            off, size, idlen = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + idlen]
            pos += 24 + idlen
            if b"gfx950" in name and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + 1)


def kernels(elf):
    """The metadata of a code object's kernels (the ELF's AMDGPU note, type 32)."""
    (shoff,) = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        h = shoff + i * shentsize
        (kind,) = struct.unpack_from("<I", elf, h + 4)
        off, size = struct.unpack_from("<QQ", elf, h + 0x18)
        if kind != 7:  # SHT_NOTE
            continue
        pos, end = off, off + size
        while pos < end:
            nlen, dlen, ntype = struct.unpack_from("<III", elf, pos)
            desc = pos + 12 + (nlen + 3) // 4 * 4
            if ntype == 32:
                yield from msgpack.unpackb(elf[desc:desc + dlen])["amdhsa.kernels"]
            pos = desc + (dlen + 3) // 4 * 4


@pytest.fixture(scope="module")
def scratch():
    import fmms_amd

    data = open(fmms_amd.LIB_PATH, "rb").read()
    return {k[".name"]: k[".private_segment_fixed_size"]
            for o in code_objects(data) for k in kernels(o)}


# the FP64 and FP32 M2L of the orders up to 10 and both P2P kernels; a few spilled
# registers are the price of an occupancy bound, an array in scratch is not
@pytest.mark.parametrize("kernels,count", [(("k_m2l", "k_m2l_shared"), 10),
                                           (("k_m2l32", "k_m2l32_staged"), 10),
                                           (("k_p2p_fp64", "k_p2p_mixed"), 2)])
def test_pair_kernels_keep_their_operands_in_registers(scratch, kernels, count):
    mine = {n: b for n, b in scratch.items() if any(f"N4fmmh{len(k)}{k}" in n and
                                                   n.split(k, 1)[1][:1] in "IE" for k in kernels)}
    assert len(mine) == count, sorted(mine)
    assert max(mine.values()) <= 16 * 4, {n: b for n, b in mine.items() if b}
