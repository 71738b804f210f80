"""Where the full-attention loop stands in the built code (no GPU needed)."""
import os
import re
import shutil
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "o1.c_amd", "libo1hip.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def code_objects(path):
    """The gfx950 code objects of a library's offload bundles."""
    data = open(path, "rb").read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        n, p = struct.unpack_from("<Q", data, at + len(magic))[0], at + len(magic) + 8
        for _ in range(n if n < 16 else 0):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in name:
                yield data[at + off:at + off + size]
        at = data.find(magic, at + 1)


@pytest.mark.skipif(not shutil.which(OBJDUMP), reason="no llvm-objdump")
def test_plain_flash_loop_position(tmp_path):
    """The key loop of the full-attention kernel starts 12 or 16 bytes past a
    32-byte boundary; elsewhere it runs 1-2 % slower. Its first instruction is the
    kernel's first three-way maximum (the softmax of the tile before)."""
    for i, co in enumerate(code_objects(LIB)):
        if b"flash_pp16_kernel" not in co:
            continue
        f = tmp_path / f"{i}.o"
        f.write_bytes(co)
        names = set(re.findall(rb"_Z17flash_pp16_kernelILi0EEv6FaArgs(?=\0)", co))
        assert names
        dis = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--disassemble-symbols=" + names.pop().decode(), str(f)],
                             check=True, capture_output=True, text=True).stdout
        loop = int(re.search(r"^\tv_max3_f32 .*// ([0-9A-F]+):", dis, re.M).group(1), 16)
        assert loop % 32 in (12, 16), hex(loop)
        return
    pytest.fail("no code object holds the attention kernel")
