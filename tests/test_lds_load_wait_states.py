"""The wait states before buffer -> LDS loads, in the built library's machine code.

The loads are inline assembly, before which the compiler inserts no wait states of its own.
gfx950 asks for one between a write of m0 and a load to LDS that uses it, and for five between
a vector instruction's write of a scalar register (v_readlane, as behind a spilled buffer
resource; v_readfirstlane; a compare) and a memory instruction that reads it.
"""
from __future__ import annotations

import pathlib
import re
import shutil
import struct
import subprocess

import pytest

from modelsharp_amd import native

OBJDUMP = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin:/opt/rocm/bin")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(lib: bytes):
    """The gfx950 code objects of the library's offload bundles (one per source file)."""
    at = lib.find(MAGIC)
    while at >= 0:
        (count,), p = struct.unpack_from("<Q", lib, at + len(MAGIC)), at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, n = struct.unpack_from("<QQQ", lib, p)
            triple, p = lib[p + 24:p + 24 + n], p + 24 + n
            if b"gfx950" in triple and size:
                yield lib[at + offset:at + offset + size]
        at = lib.find(MAGIC, at + 1)


def scalar_registers(operand: str) -> set[str]:
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    if m:
        return {f"s{i}" for i in range(int(m[1]), int(m[2]) + 1)}
    return {operand} if re.fullmatch(r"s\d+", operand) else set()


def violations(lines):
    """(function, writer, load) for each load to LDS too close behind a write of its operands."""
    function, recent, loads, found = "", [], 0, []
    for line in lines:
        if line.endswith(">:\n"):
            function, recent = line.split("<")[-1][:-3], []
            continue
        words = re.split(r"[\s,]+", line.split("//")[0].strip())
        if not words[0]:
            continue
        if words[0].startswith("buffer_load") and "lds" in words:
            loads += 1
            reads, states = set().union(*(scalar_registers(w) for w in words[1:])), 0
            for w in reversed(recent):
                if w[0].startswith("s_mov") and w[1:2] == ["m0"] and states < 1:
                    found.append((function, " ".join(w), " ".join(words)))
                if w[0].startswith(("v_readlane", "v_readfirstlane", "v_cmp")) and states < 5 and \
                        scalar_registers(w[1]) & reads:
                    found.append((function, " ".join(w), " ".join(words)))
                states += int(w[1]) + 1 if w[0] == "s_nop" else 1
        recent = recent[-7:] + [words]
    return loads, found


@pytest.mark.skipif(OBJDUMP is None, reason="llvm-objdump is not installed")
def test_lds_loads_keep_their_wait_states(tmp_path):
    lib = pathlib.Path(native.__file__).parent / "lib" / "libms_hip_nbits.so"
    total = 0
    for i, obj in enumerate(code_objects(lib.read_bytes())):
        path = tmp_path / f"object{i}"
        path.write_bytes(obj)
        with subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], stdout=subprocess.PIPE, text=True) as p:
            loads, found = violations(p.stdout)
        assert p.returncode == 0
        assert not found, f"{len(found)} loads, the first: {found[0]}"
        total += loads
    assert total > 100   # the prefill, block, W4A8 and attention kernels stage through them
