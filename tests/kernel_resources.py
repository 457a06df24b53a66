"""Registers, scratch and LDS of every kernel in the built library, from the metadata its code
objects carry (the AMDGPU note: a msgpack map)."""
import struct
import subprocess

import msgpack

from karume_amd import _ffi

_MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    at = data.find(_MAGIC)
    while at >= 0:
        (entries,) = struct.unpack_from("<Q", data, at + 24)
        cursor = at + 32
        for _ in range(entries):
            offset, size, name_len = struct.unpack_from("<QQQ", data, cursor)
            name = data[cursor + 24:cursor + 24 + name_len]
            cursor += 24 + name_len
            if name.startswith(b"hip") and size:
                yield data[at + offset:at + offset + size]
        at = data.find(_MAGIC, at + 24)


def _metadata(elf):
    (table,) = struct.unpack_from("<Q", elf, 0x28)
    entry_size, entries = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(entries):
        _, kind, _, _, offset, size = struct.unpack_from("<IIQQQQ", elf, table + i * entry_size)
        if kind != 7:   # SHT_NOTE
            continue
        at = offset
        while at < offset + size:
            name_size, desc_size, note = struct.unpack_from("<III", elf, at)
            desc = at + 12 + (name_size + 3) // 4 * 4
            if note == 32 and elf[at + 12:at + 18] == b"AMDGPU":
                return msgpack.unpackb(elf[desc:desc + desc_size])
            at = desc + (desc_size + 3) // 4 * 4
    raise AssertionError("a code object without metadata")


def kernels():
    """{demangled name: metadata} of the built library."""
    data = open(_ffi.LIB_PATH, "rb").read()
    found = {k[".name"]: k for elf in _code_objects(data) for k in _metadata(elf)["amdhsa.kernels"]}
    names = subprocess.run(["c++filt"], input="\n".join(found), capture_output=True, text=True,
                           check=True).stdout.split("\n")
    plain = (n.replace("(anonymous namespace)::", "").split("(")[0] for n in names)
    return {n.removeprefix("void "): k for n, k in zip(plain, found.values())}


def registers(kernel):
    """32-bit vector registers a lane takes; 512 a SIMD lane, shared by its waves."""
    return kernel[".vgpr_count"]   # accumulation registers included on this target


def scratch(kernel):
    return kernel[".private_segment_fixed_size"]
