"""What the compiler gave the decode kernels, from the metadata of the code objects built here: the kernels of 1-48 tokens
run without scratch memory. A register spill or a struct indexed at run time puts a chain of scratch accesses ahead of
their first loads (an adapter's module table there made the int8 (17408, 5120) product of one token 1.4x slower)."""

import os
import re
import struct

import msgpack
import pytest

from qwenny_amd.build import LIB


def _kernels(path):
    """{name: (scratch bytes, spilled VGPRs)} over the offload bundles of a shared library built by hipcc."""
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
            phoff, phentsize, phnum = struct.unpack_from("<Q", elf, 32)[0], *struct.unpack_from("<HH", elf, 54)
            for i in range(phnum):
                kind, _, off, _, _, filesz = struct.unpack_from("<IIQQQQ", elf, phoff + i * phentsize)
                if kind != 4:  # PT_NOTE
                    continue
                namesz, descsz, _ = struct.unpack_from("<III", elf, off)
                start = off + 12 + (namesz + 3) // 4 * 4
                assert start + descsz <= off + filesz
                for k in msgpack.unpackb(elf[start:start + descsz]).get("amdhsa.kernels", []):
                    out[k[".name"]] = (k[".private_segment_fixed_size"], k[".vgpr_spill_count"])
    return out


@pytest.mark.skipif(not os.path.exists(LIB), reason="nothing built")
@pytest.mark.parametrize("kernel", ["skinny_mw_kernel", "mid_kernel", "skinny_m1_kernel", "skinny_m1w_kernel",
                                    "skinny_mt_kernel"])
def test_no_scratch(kernel):
    found = {n: r for n, r in _kernels(LIB).items() if f"{len(kernel)}{kernel}I" in n}
    assert found
    assert not {n: r for n, r in found.items() if r != (0, 0)}
