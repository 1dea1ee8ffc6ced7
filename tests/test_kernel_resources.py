"""What the compiler made of the kernels: the instantiations that carry the main path keep their vector registers.

The code objects in libfp8bs.so carry notes with the registers, spills and scratch of every kernel."""
import struct
import subprocess

import pytest

msgpack = pytest.importorskip("msgpack")

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _gfx950_objects(data):
    """The gfx950 ELF images of the offload bundles in a library: after the magic the number of entries, then of each its offset from
    the magic, its size, and its target's name with the name's length ahead of it."""
    at = data.find(MAGIC)
    while at >= 0:
        entries, = struct.unpack_from("<Q", data, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        if 0 < entries < 16:
            for _ in range(entries):
                offset, size, length = struct.unpack_from("<QQQ", data, pos)
                if size and b"gfx950" in data[pos + 24:pos + 24 + length]:
                    yield data[at + offset:at + offset + size]
                pos += 24 + length
        at = data.find(MAGIC, at + 1)


def _kernels(elf):
    """The kernels' entries of the AMDGPU metadata note (owner "AMDGPU", type 32, msgpack)."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    entry, count = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, shoff + i * entry + 4)
        if kind != 7:                                                              # SHT_NOTE
            continue
        pos, size = struct.unpack_from("<QQ", elf, shoff + i * entry + 24)
        end = pos + size
        while pos < end:
            name, desc, note = struct.unpack_from("<III", elf, pos)
            body = pos + 12 + (name + 3) // 4 * 4
            if note == 32 and elf[pos + 12:pos + 12 + name].rstrip(b"\0") == b"AMDGPU":
                yield from msgpack.unpackb(elf[body:body + desc], strict_map_key=False)["amdhsa.kernels"]
            pos = body + (desc + 3) // 4 * 4


@pytest.fixture(scope="module")
def spills(pkg):
    """gemm_tr_kernel's template arguments -> vector registers that it spills."""
    with open(pkg._lib.LIB_PATH, "rb") as f:
        data = f.read()
    found = {k[".name"]: k[".vgpr_spill_count"] for elf in _gfx950_objects(data) for k in _kernels(elf)}
    names = subprocess.run(["c++filt"] + list(found), check=True, stdout=subprocess.PIPE, text=True).stdout.splitlines()
    tiled = {n.split("<")[1].split(">")[0].replace(" ", ""): v for n, v in zip(names, found.values()) if "gemm_tr_kernel<" in n}
    assert len(tiled) > 100
    return tiled


# BM, BN, WM, WN, EPI of the epilogue where there is one, stages
TILES = ["256,256,64,128,%d,%d,2", "256,192,64,96,%d,%d,2", "256,128,64,64,%d,%d,2", "256,128,64,64,%d,%d,3", "192,192,48,96,%d,%d,3",
         "128,128,64,64,%d,%d,2", "128,128,32,64,%d,%d,4", "64,256,32,64,%d,%d,3", "64,128,32,32,%d,%d,3", "64,64,32,32,%d,%d,4"]


@pytest.mark.parametrize("tile", TILES)
def test_unsplit_kernels_do_not_spill(spills, tile):
    for mode in (0, 2):                                                            # dense and grouped
        assert spills[tile % (mode, 0) + ",false,false"] == 0


def test_summed_split_of_192x192_does_not_spill(spills):
    """What it spills is reloaded ahead of the K loop and waited for inside it, by waits that drain the copies too: 4096 x 2112 x 7168 in
    two partitions took 95 us with two registers spilled, 79 with none."""
    assert spills["192,192,48,96,4,0,3,false,false"] == 0
