"""Register use of kernels whose speed hangs on it, read from the metadata that the
compiler writes into the library built here (no GPU)."""
import struct

import msgpack
import pytest


def code_objects(data):
    """The gfx950 ELF images in the library's offload bundles."""
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := data.find(magic, at)) >= 0:
        n, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in name:
                yield data[at + off:at + off + size]
        at += 24


def kernels(elf):
    """name -> metadata of an image's kernels (its NT_AMDGPU_METADATA note)."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        typ, = struct.unpack_from("<I", elf, shoff + i * shentsize + 4)
        off, size = struct.unpack_from("<QQ", elf, shoff + i * shentsize + 24)
        if typ != 7:  # SHT_NOTE
            continue
        namesz, descsz, ntype = struct.unpack_from("<III", elf, off)
        if ntype == 32:
            desc = off + 12 + (namesz + 3) // 4 * 4
            for k in msgpack.unpackb(elf[desc:desc + descsz])["amdhsa.kernels"]:
                yield k[".name"], k


@pytest.fixture(scope="module")
def found():
    from cosxamix_amd import _lib
    _lib.load()
    return {n: k for e in code_objects(open(_lib.LIB_PATH, "rb").read()) for n, k in kernels(e)}


def test_the_row_norms_keep_their_waves(found):
    # 72 registers are seven waves a SIMD. With the ordered sum's squares kept in
    # registers they had 98, four waves, for every row of a launch (8000 rows of
    # 2048 values 38 -> 42 us, of 896 19 -> 25)
    norms = {n: k for n, k in found.items()
             if any(s in n for s in ("k_rmsnormI", "k_norm_rowsI", "k_norm_quant"))}
    assert len(norms) == 12
    for n, k in norms.items():
        assert k[".vgpr_count"] <= 72, (n, k[".vgpr_count"])
        assert k[".private_segment_fixed_size"] == 0, n
