"""The compiled kernels save no vector register under a narrower EXEC mask
than the one it is reloaded under.

Where two branches of a wavefront meet, the block starts with the instruction
that brings the other lanes back (s_or_b64 exec, s_andn2_saveexec_b64, ...).
The register allocator puts its copies and spills behind it, unless a scalar
instruction that it placed at the block's top comes first: then they run for
one side's lanes only, and a later reload gives the other side's lanes what the
register held before.  Kernels near the register limit were built so: phase
equilibrium by teams of 8 at Nc = 11 then lost the interaction coefficients of
half the lanes, and with them phases.  build.py's flags keep such scalar
instructions away; this test reads the built code for what they miss: a block
entered by a branch on EXEC = 0 that begins with nothing but copies and spills
of vector registers up to the instruction that restores EXEC."""
import os
import re
import struct
import subprocess

import pytest

from opencaeporox_amd import abi

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"

RESTORE = re.compile(r"s_or_b64 exec, exec|s_andn2_saveexec_b64|s_or_saveexec_b64")
COPY = re.compile(r"v_accvgpr_|scratch_(load|store)_|buffer_(load|store)_|v_mov_b(32|64)_e32")
SCALAR = re.compile(r"s_waitcnt|s_nop|s_mov|v_readlane_b32|v_writelane_b32")


def suspects(lines):
    """(address, instructions) of the blocks described above, from a disassembly."""
    code, targets, base, pc = [], set(), 0, None
    for line in lines:
        m = re.match(r"([0-9a-f]+) <(.+)>:", line)
        if m:
            base = int(m.group(1), 16)
            continue
        m = re.match(r"\t(\S.*?)\s*// ([0-9A-F]+):", line)
        if not m:
            continue
        text, at = m.group(1), int(m.group(2), 16)
        code.append((at, text))
        if text.startswith("s_cbranch_execz"):
            off = re.search(r"<[^>]*?\+0x([0-9a-f]+)>\s*$", line)
            targets.add(base + int(off.group(1), 16) if off else base)
        # a branch out of the 16-bit range: getpc, add an offset, setpc
        if text.startswith("s_getpc_b64"):
            pc = at + 4
        elif pc is not None and text.startswith("s_add_u32"):
            off = text.split(",")[-1].strip()
            if re.fullmatch(r"(0x[0-9a-f]+|-?\d+)", off):
                off = int(off, 0)
                targets.add(pc + (off - (1 << 32) if off >= 1 << 31 else off))
            pc = None
    found, copies, at0 = [], None, 0
    for at, text in code:
        if at in targets:
            copies, at0 = [], at
        if copies is None:
            continue
        if RESTORE.match(text):
            if copies:
                found.append((at0, copies))
            copies = None
        elif COPY.match(text):
            copies.append(text)
        elif not SCALAR.match(text):
            copies = None
    return found


def test_the_check_finds_a_save_ahead_of_the_restore():
    dis = ["0000000000001000 <k>:",
           "\ts_and_saveexec_b64 s[0:1], vcc                  // 000000001000: BE80206A ",
           "\ts_cbranch_execz 3                               // 000000001004: BF880003 <k+0x14>",
           "\tv_add_f64 v[2:3], v[2:3], v[4:5]                // 000000001008: D2800002 ",
           "\tv_add_f64 v[2:3], v[2:3], v[4:5]                // 000000001010: D2800002 "]
    late = ["\ts_movk_i32 s22, 0x204                           // 000000001018: B0160204 ",
            "\ts_andn2_saveexec_b64 s[0:1], s[24:25]           // 00000000101C: BE802318 "]
    save = "\tv_accvgpr_write_b32 a28, v196                   // 000000001014: D3D94018 "
    assert suspects(dis + [save] + late) == [(0x1014, ["v_accvgpr_write_b32 a28, v196"])]
    # the save behind the restore, and a restore alone
    assert suspects(dis + [late[1].replace("00101C", "001014"), save.replace("001014", "001018")]) == []
    # a branch's own work ahead of the restore
    assert suspects(dis + [save.replace("v_accvgpr_write_b32 a28, v196", "ds_write_b64 v1, v[2:3]      ")] + late) == []


def test_no_vector_save_ahead_of_the_exec_restore():
    if not os.path.exists(OBJDUMP):
        pytest.skip("no disassembler")
    with open(abi.LIB_PATH, "rb") as f:
        blob = f.read()
    found, objects = [], 0
    start = blob.find(MAGIC)
    while start >= 0:
        n, = struct.unpack_from("<Q", blob, start + len(MAGIC))
        p = start + len(MAGIC) + 8
        for _ in range(n):
            off, size, ln = struct.unpack_from("<QQQ", blob, p)
            name = blob[p + 24:p + 24 + ln].decode()
            p += 24 + ln
            if "gfx950" in name and size:
                objects += 1
                found += _code_object(blob[start + off:start + off + size])
        start = blob.find(MAGIC, p)
    assert objects >= 9, "one code object per kernel source"
    assert not found, "\n".join(f"{at:#x}: {len(c)} copies, {c[:3]}" for at, c in found[:10])


def _code_object(elf):
    import tempfile
    with tempfile.NamedTemporaryFile(suffix=".co") as f:
        f.write(elf)
        f.flush()
        with subprocess.Popen([OBJDUMP, "-d", f.name], stdout=subprocess.PIPE, text=True) as p:
            out = suspects(p.stdout)
        assert p.returncode == 0
    return out
