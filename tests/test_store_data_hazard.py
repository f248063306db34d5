"""A 16-byte store reads its data registers a little after it has been issued, so that what follows must leave them alone for a while.  The library's
own device code is disassembled and every such store looked at: how many wait states lie between it and the first VALU write of a register it
stores.  Two where the store has no scalar offset, which the compiler sees to; four where it has one: there the compiler leaves none, and
with none the tile kernels stored new values now and then (store_c in common.hpp)."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "hipkittensp_amd", "libmxfp6_gemm.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(data):
    at = data.find(MAGIC)
    while at >= 0:
        (n,), p = struct.unpack_from("<Q", data, at + 24), at + 32
        for _ in range(n):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24 : p + 24 + length] and size:
                yield data[at + offset : at + offset + size]
            p += 24 + length
        at = data.find(MAGIC, at + 24)


def registers(operand):
    m = re.fullmatch(r"([va])(?:\[(\d+):(\d+)\]|(\d+))", operand)
    return set() if not m else {(m[1], i) for i in (range(int(m[2]), int(m[3]) + 1) if m[2] else [int(m[4])])}


def distances(listing):
    """(has a scalar offset, wait states up to 8, instruction) of every 16-byte vector store, in the order of the code and past branches that are not taken."""
    code = []
    for line in listing.splitlines():
        m = re.match(r"\s+([a-z_0-9]+)\s*(.*?)\s*(//.*)?$", line)
        code.append((m[1], [x.strip() for x in m[2].split(",")]) if m else ("", []))
    for i, (op, args) in enumerate(code):
        if not re.match(r"(buffer|global|flat)_store_dwordx[34]$", op):
            continue
        buffer = op.startswith("buffer")
        data = registers(args[0] if buffer else args[1])
        assert data, (op, args)
        scalar = buffer and re.match(r"(s\d|m0|ttmp)", args[3].split()[0] if len(args) > 3 else "") is not None
        states = 0
        for nxt, a in code[i + 1 : i + 9]:
            if nxt in ("", "s_endpgm"):
                states = 8
            elif nxt.startswith("v_") and not nxt.startswith("v_cmp") and data & (registers(a[0]) | (registers(a[1]) if "swap" in nxt else set())):
                break
            states += int(a[0], 0) + 1 if nxt == "s_nop" else 1
            if states >= 8:
                break
        yield scalar, min(states, 8), f"{op} {', '.join(args)}"


def test_listing_is_understood():
    text = """
\tbuffer_store_dwordx4 v[0:3], v66, s[8:11], s0 offen nt     // 1:
\tv_mov_b32_e32 v2, v9     // 2:
\tglobal_store_dwordx4 v[6:7], v[2:5], off     // 3:
\ts_nop 0     // 4:
\ts_mov_b32 s1, s2     // 5:
\tv_permlane16_swap_b32_e32 v70, v5     // 6:
\tbuffer_store_dwordx4 v[0:3], v66, s[8:11], 0 offen     // 7:
\ts_nop 3     // 8:
\tv_mov_b32_e32 v3, v9     // 9:
"""
    assert [d[:2] for d in distances(text)] == [(True, 0), (False, 2), (False, 4)]


def test_stored_registers_are_left_alone(tmp_path):
    if not os.path.exists(LIB) or not os.path.exists(OBJDUMP):
        pytest.skip("the library is not built, or no disassembler")
    data = open(LIB, "rb").read()
    seen = {False: 0, True: 0}
    for n, co in enumerate(code_objects(data)):
        f = tmp_path / f"{n}.co"
        f.write_bytes(co)
        listing = subprocess.check_output([OBJDUMP, "-d", "--no-show-raw-insn", str(f)], text=True)
        for scalar, states, what in distances(listing):
            seen[scalar] += 1
            assert states >= (4 if scalar else 2), (n, what, states)
    assert min(seen.values()) > 1000, seen
