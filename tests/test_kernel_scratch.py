"""No kernel of the built library keeps private memory (scratch): a launch reserves it for every lane of the card, and
what lands there is memory traffic that no source line shows."""
import struct

import msgpack

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    """The AMDGPU ELF images of the offload bundles in a host library."""
    at = data.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"amdgcn" in name and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + len(MAGIC))


def _kernels(elf):
    """The kernel entries of a code object's metadata note (NT_AMDGPU_METADATA, msgpack)."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    entsize, count = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(count):
        _, kind, _, _, off, size = struct.unpack_from("<IIQQQQ", elf, shoff + i * entsize)
        at, end = off, off + size
        while kind == 7 and at < end:  # SHT_NOTE
            namesz, descsz, ntype = struct.unpack_from("<III", elf, at)
            desc = at + 12 + -(-namesz // 4) * 4
            if ntype == 32:
                yield from msgpack.unpackb(elf[desc:desc + descsz], strict_map_key=False)["amdhsa.kernels"]
            at = desc + -(-descsz // 4) * 4


def test_no_kernel_uses_scratch():
    from leankv_amd.build import LIB_PATH

    with open(LIB_PATH, "rb") as f:
        kernels = [k for elf in _code_objects(f.read()) for k in _kernels(elf)]
    assert any("bulk_update_kernel" in k[".name"] for k in kernels) and len(kernels) > 50
    used = {k[".name"]: k[".private_segment_fixed_size"] for k in kernels if k[".private_segment_fixed_size"]}
    assert not used
