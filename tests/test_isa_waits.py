"""Wait states that gfx950 asks the program for, in the built library's own code.

The compiler inserts them for the instructions it emits, but does not look
into inline assembly, where the LDS-DMA copies (csrc/common.hpp) stand:

  * an SALU write of m0, then an LDS-DMA load: one wait state;
  * a VALU write of an SGPR (v_readlane of a spilled address, say), then a
    vector-memory instruction that reads it: five.

Both are silent where broken: a copy lands at the previous copy's LDS address,
or reads from a stale base."""
import os
import re
import struct
import subprocess

import pytest

LIBRARY = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "omni-rs_amd", "libomni_int8.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
M0_WAIT, SGPR_WAIT = 1, 5


def code_objects(data):
    """The gfx950 ELF images of the library's offload bundles."""
    at = data.find(MAGIC)
    while at >= 0:
        pos = at + len(MAGIC) + 8
        for _ in range(struct.unpack_from("<Q", data, at + len(MAGIC))[0]):
            offset, size, name = struct.unpack_from("<QQQ", data, pos)
            if b"gfx950" in data[pos + 24:pos + 24 + name]:
                yield data[at + offset:at + offset + size]
            pos += 24 + name
        at = data.find(MAGIC, at + 1)


def sgprs(operand):
    m = re.match(r"s\[(\d+):(\d+)\]|s(\d+)\b", operand)
    if not m:
        return ()
    return range(int(m[1]), int(m[2]) + 1) if m[1] else (int(m[3]),)


def broken_waits(listing):
    """(copies seen, [what is broken]) of a disassembly."""
    copies, broken, kernel = 0, [], ""
    valu, m0, now = {}, -99, 0  # SGPR -> when a VALU wrote it last, the same for m0 and SALU
    for line in listing.splitlines():
        label = re.match(r"[0-9a-f]+ <(.*)>:", line)
        if label:
            kernel = label[1]
            continue
        parts = line.split("//")[0].split(None, 1)
        if not parts or not re.match(r"[a-z]+_", parts[0]):
            continue
        op, args = parts[0], [a.strip() for a in parts[1].split(",")] if len(parts) > 1 else []
        if re.match(r"(global|buffer|flat|scratch)_", op):
            if "_lds_" in op:
                copies += 1
                if now - m0 < M0_WAIT:
                    broken.append(f"{kernel}: m0, then {line.strip()}")
            for a in args:
                for r in sgprs(a):
                    if now - valu.get(r, -99) < SGPR_WAIT:
                        broken.append(f"{kernel}: s{r} of a VALU, then {line.strip()}")
        now += 1 + (int(args[0], 0) if op == "s_nop" else 0)
        # The second operand of carries, wide multiply-adds and divide scales is written, too.
        wide = re.search(r"_co_|mad_[iu]64|div_scale", op)
        for a in args[:2] if wide else args[:1]:
            for r in sgprs(a):
                if op.startswith("v_"):
                    valu[r] = now
                elif not op.startswith(("global", "buffer", "flat", "scratch", "ds_")):
                    valu.pop(r, None)
        if op.startswith("s_") and args and args[0] == "m0":
            m0 = now
    return copies, broken


def test_the_check_sees_a_missing_wait():
    assert broken_waits("s_mov_b32 m0, s4\nglobal_load_lds_dwordx4 v1, s[2:3]")[1]
    assert not broken_waits("s_mov_b32 m0, s4\ns_nop 0\nglobal_load_lds_dwordx4 v1, s[2:3]")[1]
    late = "v_readlane_b32 s3, v9, 1\ns_mov_b32 m0, s4\ns_nop %d\nglobal_load_lds_dwordx4 v1, s[2:3]"
    assert broken_waits(late % 2)[1] and not broken_waits(late % 3)[1]
    assert not broken_waits("v_readlane_b32 s3, v9, 1\ns_mov_b64 s[2:3], s[2:3]\nglobal_load_dword v1, v2, s[2:3]")[1]


def test_library_waits_before_its_copies(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    with open(LIBRARY, "rb") as f:
        images = list(code_objects(f.read()))
    assert images
    copies = 0
    for i, image in enumerate(images):
        path = tmp_path / f"{i}.co"
        path.write_bytes(image)
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--mcpu=gfx950", str(path)], check=True,
                                 capture_output=True, text=True).stdout
        n, broken = broken_waits(listing)
        copies += n
        assert not broken, f"{len(broken)} missing waits, the first: {broken[0]}"
    assert copies > 1000
