"""Register spills of the built kernels, from the code objects' own metadata."""
import struct
from pathlib import Path

import msgpack
import pytest

from trifuse_amd import _lib, build

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _gpu_images(lib: bytes):
    """The gfx950 ELF images of a HIP library: bundles of (offset, size, target) entries."""
    at = lib.find(MAGIC)
    while at >= 0:
        n = struct.unpack_from("<Q", lib, at + len(MAGIC))[0]
        pos = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", lib, pos)
            target = lib[pos + 24:pos + 24 + idlen]
            pos += 24 + idlen
            if build.ARCH.encode() in target and size:
                yield lib[at + off:at + off + size]
        at = lib.find(MAGIC, at + 1)


def _kernels(elf: bytes):
    """amdhsa.kernels of an image's metadata note (type 32, msgpack)."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        kind, = struct.unpack_from("<I", elf, shoff + i * shentsize + 4)
        off, size = struct.unpack_from("<QQ", elf, shoff + i * shentsize + 24)
        pos = off
        while kind == 7 and pos < off + size:
            name, desc, note = struct.unpack_from("<III", elf, pos)
            body = pos + 12 + (name + 3) // 4 * 4
            if note == 32:
                yield from msgpack.unpackb(elf[body:body + desc])["amdhsa.kernels"]
            pos = body + (desc + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    data = Path(_lib.LIB_PATH).read_bytes()
    return {k[".name"]: k for image in _gpu_images(data) for k in _kernels(image)}


# A tile's accumulators, raw weights and fragments fill its registers to the
# bound of its launch; a spilled one is reloaded in the main loop.
def test_register_kernels_keep_their_registers(kernels):
    wr = {n: k for n, k in kernels.items() if "ggemm_wr_kernel" in n}
    assert len(wr) >= 50  # modes x storage types x code widths x tiles
    bad = {n: (k[".vgpr_spill_count"], k[".private_segment_fixed_size"]) for n, k in wr.items()
           if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]}
    assert not bad
