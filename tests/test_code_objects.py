"""The machine code of the built library, kernel by kernel.

A 64-bit shift by a vector register reads that register and the next one.  When
the amount is in the last register that a wave has, the next one belongs to
nobody or to another wave, and the shift now and then comes out wrong (known
from the gfx90a generation, where the compiler avoids it; on gfx950 it does
not).  Nothing shows in the source, so the built code is looked at."""
from __future__ import annotations

import os
import re
import shutil
import struct
import subprocess

import pytest

from immunodbscan_amd import _lib

LLVM = "/opt/rocm/llvm/bin"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
SHIFT = re.compile(r"\bv_(?:lshlrev_b64|lshrrev_b64|ashrrev_i64)(?:_e64)? v\[\d+:\d+\], v(\d+),")
REGISTER_BLOCK = 8  # registers are given to a wave in blocks


def code_objects():
    data = open(_lib.LIB_PATH, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        n = struct.unpack_from("<Q", data, at + len(MAGIC))[0]
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, name = struct.unpack_from("<QQQ", data, p)
            p += 24
            if b"gfx950" in data[p:p + name]:
                yield data[at + off:at + off + size]
            p += name
        at = data.find(MAGIC, at + 1)


def last_register_shifts(asm: str, registers: dict[str, int]) -> list[str]:
    found, kernel = [], None
    for line in asm.splitlines():
        m = re.match(r"^[0-9a-f]+ <(\S+)>:", line)
        if m:
            kernel = m.group(1)
        m = SHIFT.search(line)
        if m and kernel in registers:
            blocks = -(-registers[kernel] // REGISTER_BLOCK)
            if int(m.group(1)) == blocks * REGISTER_BLOCK - 1:
                found.append(f"{kernel} ({registers[kernel]} registers): {line.strip()}")
    return found


def test_the_check_finds_such_a_shift():
    asm = "0000 <k>:\n v_lshrrev_b64 v[4:5], v31, v[4:5]\n v_lshlrev_b64 v[4:5], s3, v[4:5]\n v_lshlrev_b64 v[4:5], v7, v[4:5]"
    assert len(last_register_shifts(asm, {"k": 32})) == 1
    assert len(last_register_shifts(asm, {"k": 30})) == 1
    assert not last_register_shifts(asm, {"k": 33})


@pytest.mark.skipif(not shutil.which(os.path.join(LLVM, "llvm-objdump")), reason="no LLVM tools")
def test_no_shift_amount_in_the_last_register(tmp_path):
    kernels, shifts, found = 0, 0, []
    for i, obj in enumerate(code_objects()):
        path = str(tmp_path / f"{i}.elf")
        open(path, "wb").write(obj)
        notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", path], capture_output=True, text=True,
                               check=True).stdout
        registers = {}
        for block in notes.split("- .agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(\S+)", block)
            count = re.search(r"\.vgpr_count:\s+(\d+)", block)
            registers[name.group(1)] = int(count.group(1))
        asm = subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", "--no-show-raw-insn", path], capture_output=True,
                             text=True, check=True).stdout
        kernels += len(registers)
        shifts += len(SHIFT.findall(asm))
        found += last_register_shifts(asm, registers)
    print(f"{kernels} kernels, {shifts} shifts by a register")
    assert kernels > 100
    assert not found, "\n".join(found)
