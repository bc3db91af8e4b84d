"""Register and scratch use of the built kernels, read from the metadata notes
of libkxw4.so's own code objects (no GPU needed)."""
import struct

import msgpack
import pytest

from knivesysl_xe_amd import _lib

BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"
NT_AMDGPU_METADATA = 32


def code_objects(blob):
    """The gfx950 ELF images of every offload bundle in `blob`."""
    at = blob.find(BUNDLE)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", blob, at + len(BUNDLE))
        p = at + len(BUNDLE) + 8
        for _ in range(count):
            offset, size, id_len = struct.unpack_from("<QQQ", blob, p)
            if b"gfx950" in blob[p + 24:p + 24 + id_len]:
                yield blob[at + offset:at + offset + size]
            p += 24 + id_len
        at = blob.find(BUNDLE, at + 1)


def kernels(elf):
    """The kernel records of a code object's metadata note."""
    (shoff,) = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        sh_type, _, _, offset, size = struct.unpack_from("<IQQQQ", elf, shoff + i * shentsize + 4)
        if sh_type != 7:                                 # SHT_NOTE
            continue
        p = offset
        while p < offset + size:
            namesz, descsz, kind = struct.unpack_from("<III", elf, p)
            desc = p + 12 + (namesz + 3) // 4 * 4
            if kind == NT_AMDGPU_METADATA:
                yield from msgpack.unpackb(elf[desc:desc + descsz], strict_map_key=False)["amdhsa.kernels"]
            p = desc + (descsz + 3) // 4 * 4


@pytest.fixture(scope="module")
def records():
    with open(_lib.LIB_PATH, "rb") as f:
        return [k for elf in code_objects(f.read()) for k in kernels(elf)]


def test_strip_kernel_keeps_nothing_in_scratch(records):
    # a value kept in private memory is stored and waited for between the
    # first two stages' loads, which are meant to be in flight together
    strip = [k for k in records if "strip_kernel" in k[".name"]]
    assert len(strip) > 40
    bad = {k[".name"]: k[".private_segment_fixed_size"] for k in strip if k[".private_segment_fixed_size"]}
    assert not bad
