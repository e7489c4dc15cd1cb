"""Placement of the one-row decode step's kernels in the gfx950 code object:
the names of csrc/decode_step.order, in that order and without another kernel
between them."""
import os
import struct

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "dolittle_amd", "libdlhip.so")
ORDER = os.path.join(ROOT, "dolittle_amd", "csrc", "decode_step.order")
EM_AMDGPU, SHT_SYMTAB, SHT_DYNSYM, STT_FUNC = 224, 2, 11, 2


def functions(image):
    """{name: (address, size)} of one ELF64 image's functions."""
    shoff, shentsize, shnum = struct.unpack_from("<Q", image, 40)[0], *struct.unpack_from("<HH", image, 58)
    sections = [struct.unpack_from("<IIQQQQIIQQ", image, shoff + i * shentsize) for i in range(shnum)]
    found = {}
    for _, kind, _, _, offset, size, link, _, _, entry in sections:
        if kind not in (SHT_SYMTAB, SHT_DYNSYM):
            continue
        strings = sections[link][4]
        for at in range(offset, offset + size, entry):
            name, info, _, _, value, length = struct.unpack_from("<IBBHQQ", image, at)
            if info & 15 == STT_FUNC and length:
                end = image.index(b"\0", strings + name)
                found[image[strings + name:end].decode()] = (value, length)
    return found


def code_objects(path):
    with open(path, "rb") as f:
        data = f.read()
    at = data.find(b"\x7fELF", 1)
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == EM_AMDGPU:
            yield functions(data[at:])
        at = data.find(b"\x7fELF", at + 1)


def test_step_kernels_lie_together():
    if not os.path.exists(LIB):
        pytest.skip("libdlhip.so not built")
    with open(ORDER) as f:
        wanted = [line.strip() for line in f if line.strip() and not line.startswith("#")]
    assert len(wanted) == len(set(wanted)) == 10
    holders = [found for found in code_objects(LIB) if wanted[0] in found]
    assert len(holders) == 1
    by_address = sorted(holders[0], key=lambda name: holders[0][name][0])
    assert by_address[:len(wanted)] == wanted
