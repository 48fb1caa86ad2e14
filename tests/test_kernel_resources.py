"""What the compiler gave the decode kernels, from the kernel descriptors of the code objects built here: the kernels of 1-48 tokens
run without scratch memory. A register spill or a struct indexed at run time puts a chain of scratch accesses ahead of
their first loads (an adapter's module table there made the int8 (17408, 5120) product of one token 1.4x slower)."""

import os
import re
import struct

import pytest

from qwenny_amd.build import LIB


def _kernels(path):
    """{name: scratch bytes} over the offload bundles of a shared library built by hipcc, from the kernel descriptors
    (symbols NAME.kd: u32 LDS bytes, u32 scratch bytes per lane, ..)."""
    with open(path, "rb") as f:
        data = f.read()
    out = {}
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        at = m.start()
        count, pos = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(count):
            offset, size, n = struct.unpack_from("<QQQ", data, pos)
            triple = data[pos + 24:pos + 24 + n]
            pos += 24 + n
            if b"amdgcn" not in triple or size == 0:
                continue
            elf = data[at + offset:at + offset + size]
            assert elf[:4] == b"\x7fELF"
            shoff, shentsize, shnum = struct.unpack_from("<Q", elf, 40)[0], *struct.unpack_from("<HH", elf, 58)
            # type, flags, address, offset, size, link of each section
            sections = [struct.unpack_from("<IQQQQI", elf, shoff + i * shentsize + 4) for i in range(shnum)]
            for kind, _, _, off, size, link in sections:
                if kind != 11:  # SHT_DYNSYM
                    continue
                names = sections[link][3]
                for sym in range(off, off + size, 24):
                    name, _, _, index, value, _ = struct.unpack_from("<IBBHQQ", elf, sym)
                    name = elf[names + name:elf.index(b"\0", names + name)].decode()
                    if name.endswith(".kd"):
                        at_kd = value - sections[index][2] + sections[index][3]
                        out[name[:-3]] = struct.unpack_from("<I", elf, at_kd + 4)[0]
    return out


@pytest.mark.skipif(not os.path.exists(LIB), reason="nothing built")
@pytest.mark.parametrize("kernel", ["skinny_mw_kernel", "mid_kernel", "skinny_m1_kernel", "skinny_m1w_kernel",
                                    "skinny_mt_kernel"])
def test_no_scratch(kernel):
    found = {n: r for n, r in _kernels(LIB).items() if f"{len(kernel)}{kernel}I" in n}
    assert found
    assert not {n: r for n, r in found.items() if r}
