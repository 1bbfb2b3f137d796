"""A vector store of more than eight bytes still reads its data registers while the next two instructions run: a vector
instruction that writes one of them by then changes what is stored.  The compiler keeps the two apart within a block, but was seen to
leave one instruction between them across a branch.  Every such store of the built library, followed through both
sides of branches."""
import os
import re
import struct
import subprocess

import pytest

from llmxabe_amd import _ffi
from test_spilled_registers import _code_objects

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
WAIT_STATES = 2
HEAD = re.compile(r"^([0-9a-f]+) <(.+)>:")
LINE = re.compile(r"^\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+):(?:.*<(.+?)(?:\+0x([0-9a-f]+))?>)?")
STORE = re.compile(r"(?:global|flat|buffer|scratch)_store_(?:dwordx[34]|b96|b128)$")


def _registers(operand):
    """The vector registers an operand names."""
    m = re.match(r"v\[(\d+):(\d+)\]$|v(\d+)$", operand.strip())
    if not m:
        return range(0)
    return range(int(m[1]), int(m[2]) + 1) if m[1] else range(int(m[3]), int(m[3]) + 1)


def _instructions(text):
    """[(kernel, mnemonic, operands, branch target's index or None)]"""
    base, found, kernel = {}, [], None
    for line in text.split("\n"):
        head = HEAD.match(line)
        if head:
            kernel = head[2]
            base[kernel] = int(head[1], 16)
            continue
        m = LINE.match(line)
        if m:
            target = (m[4], int(m[5] or "0", 16)) if m[4] and "branch" in m[1] else None
            found.append((kernel, m[1], m[2].split(","), int(m[3], 16), target))
    at = {address: i for i, (_, _, _, address, _) in enumerate(found)}
    return [(k, op, args, at.get(base[t[0]] + t[1]) if t and t[0] in base else None) for k, op, args, _, t in found]


def _overwritten(code, i, data, left):
    """Whether a vector instruction within `left` wait states of index `i` writes one of `data`."""
    while left > 0 and i < len(code):
        _, op, args, target = code[i]
        if op.startswith("s_endpgm"):
            return None
        if op.startswith("v_") and set(_registers(args[0])) & data:
            return i
        left -= int(args[0]) + 1 if op == "s_nop" else 1
        if target is not None:
            hit = _overwritten(code, target, data, left)
            if hit is not None or op == "s_branch":
                return hit
        i += 1
    return None


def test_the_rule_finds_what_it_is_for():
    text = """0000000000000000 <k>:
	global_store_dwordx4 v[0:1], v[4:7], off                   // 000000000000: 00000000 00000000
	s_cbranch_scc1 2                                           // 000000000008: 00000000 <k+0x14>
	s_nop 1                                                    // 00000000000C: 00000000
	v_mov_b32_e32 v4, 0                                        // 000000000010: 00000000
	v_mov_b32_e32 v7, 0                                        // 000000000014: 00000000
	s_endpgm                                                   // 000000000018: 00000000
"""
    code = _instructions(text)
    assert _overwritten(code, 1, set(range(4, 8)), WAIT_STATES) == 4   # over the branch; past the s_nop there are three
    assert _overwritten(code, 2, set(range(4, 8)), WAIT_STATES) is None
    assert _overwritten(code, 1, set(range(8, 12)), WAIT_STATES) is None


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="needs the ROCm toolchain's disassembler")
def test_no_wide_store_loses_its_registers(tmp_path):
    _ffi.lib()
    blob = open(_ffi.LIB_PATH, "rb").read()
    stores, bad = 0, []
    for n, start in enumerate(_code_objects(blob)):
        sections, = struct.unpack_from("<Q", blob, start + 40)
        size, count = struct.unpack_from("<HH", blob, start + 58)
        path = tmp_path / f"{n}.elf"
        path.write_bytes(blob[start:start + sections + size * count])
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], capture_output=True, text=True, check=True).stdout
        code = _instructions(text)
        for i, (kernel, op, args, _) in enumerate(code):
            if not STORE.match(op):
                continue
            stores += 1
            data = args[0 if op.startswith("buffer") else 1]
            data = set(_registers(data))
            assert len(data) >= 3, (op, args)
            hit = _overwritten(code, i + 1, data, WAIT_STATES)
            if hit is not None:
                bad.append((kernel, i, op, args, code[hit][1:3]))
    assert stores > 100
    assert not bad, bad[:5]
