"""What the compiler says of the kernels in the built library: the metadata that each code object carries.

Every translation unit's device code is in the library as one offload bundle: the magic, a count, and per entry an offset, a size
and a target's name; the gfx950 entries are ELF files whose AMDGPU note (type 32) is a msgpack map that lists the kernels."""
import os
import struct

import msgpack

LIBRARY = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cuv_amd", "lib", "libcuvdia.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, name = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + name] and data[at + offset:at + offset + 4] == b"\x7fELF":
                yield data[at + offset:at + offset + size]
            p += 24 + name
        at = data.find(MAGIC, at + 1)


def _notes(elf):
    headers, = struct.unpack_from("<Q", elf, 40)
    size, count = struct.unpack_from("<HH", elf, 58)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, headers + i * size + 4)
        offset, length = struct.unpack_from("<QQ", elf, headers + i * size + 24)
        p = offset
        while kind == 7 and p < offset + length:         # SHT_NOTE
            name, desc, note = struct.unpack_from("<III", elf, p)
            p += 12 + (name + 3) // 4 * 4
            if note == 32:
                yield msgpack.unpackb(elf[p:p + desc], raw=False, strict_map_key=False)
            p += (desc + 3) // 4 * 4


def kernels(library=LIBRARY):
    """{mangled name: its metadata (".vgpr_spill_count", ".private_segment_fixed_size", ...)}"""
    with open(library, "rb") as f:
        data = f.read()
    return {k[".name"]: k for elf in _code_objects(data) for note in _notes(elf) for k in note["amdhsa.kernels"]}


def preloaded(library=LIBRARY):
    """{mangled name: dwords of its arguments that come in registers}: bytes 58 and 59 of the descriptor `name`.kd, their low 7 bits"""
    with open(library, "rb") as f:
        data = f.read()
    out = {}
    for elf in _code_objects(data):
        table, = struct.unpack_from("<Q", elf, 40)
        size, count = struct.unpack_from("<HH", elf, 58)
        sections = [struct.unpack_from("<IIQQQQIIQQ", elf, table + i * size) for i in range(count)]
        for _, kind, _, _, offset, length, strings, _, _, entry in sections:
            if kind != 11:                               # SHT_DYNSYM
                continue
            for at in range(offset, offset + length, entry):
                name, _, _, section, value, _ = struct.unpack_from("<IBBHQQ", elf, at)
                start = sections[strings][4] + name
                symbol = elf[start:elf.index(b"\0", start)].decode()
                if symbol.endswith(".kd"):
                    _, _, _, address, place, _, _, _, _, _ = sections[section]
                    out[symbol[:-3]] = struct.unpack_from("<H", elf, place + value - address + 58)[0] & 127
    return out
