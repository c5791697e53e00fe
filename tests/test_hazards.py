"""Wait states that the hardware does not keep by itself, in the built kernels: the compiler spaces its own instructions and does not
look into inline assembly.  Reads the disassembly of libdistca_ca.so's own code objects; runs without a GPU."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from distca_amd._build import LIB_PATH

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(path):
    """The gfx950 code objects in the library's offload bundles."""
    data = open(path, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + idlen].decode()
            p += 24 + idlen
            if "gfx950" in name and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + 1)


def scalars(operand):
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.fullmatch(r"s(\d+)", operand)
    return {int(m[1])} if m else ({"m0"} if operand == "m0" else set())


def operands(line):
    rest = line.split(None, 1)
    return [o.strip().split()[0] for o in rest[1].split(",")] if len(rest) > 1 else []


def violations(lines):
    """(what, wait states between, instruction before, instruction) of straight-line code.  A vector instruction's write of a scalar register
    and a vector memory instruction that reads it: 5, unless a scalar instruction that uses the register, and waits for it, stands between;
    a write of M0 and a load to LDS: 1."""
    out = []
    for i, line in enumerate(lines):
        if not re.match(r"(global|buffer|flat|scratch)_(load|store|atomic)", line):
            continue
        reads = set().union(*map(scalars, operands(line)))
        to_lds = "_lds_" in line or line.endswith(" lds")
        waits = 0
        for before in reversed(lines[max(i - 5, 0):i]):
            op, ops = before.split()[0], operands(before)
            if op.startswith("v_") and ops and scalars(ops[0]) & reads:
                out.append(("scalar register", waits, before, line))
            if to_lds and waits < 1 and ops[:1] == ["m0"]:
                out.append(("M0", waits, before, line))
            if op in ("s_branch", "s_endpgm", "s_setpc_b64"):   # nothing falls through
                break
            if op.startswith("s_"):
                reads -= set().union(*map(scalars, ops)) if ops else set()
            waits += int(ops[0], 0) + 1 if op == "s_nop" else 1
            if waits >= 5:
                break
    return out


def test_hazards_planted_in_a_listing_are_found():
    load = "global_load_lds_dwordx4 v1, s[0:1] offset:2048"
    assert violations(["v_readlane_b32 s1, v252, 18", load])
    assert violations(["v_readfirstlane_b32 s0, v2", "s_nop 1", "s_mov_b32 m0, s3", "s_nop 0", load])
    assert violations(["s_mov_b32 m0, s3", load]) and not violations(["s_mov_b32 m0, s3", "s_nop 0", load])
    assert not violations(["v_readfirstlane_b32 s0, v2", "s_nop 4", load])
    assert not violations(["v_readfirstlane_b32 s0, v2", "s_mov_b64 s[0:1], s[0:1]", load])
    assert not violations(["v_readfirstlane_b32 s2, v2", "s_mov_b32 m0, s3", "s_nop 0", load])


@pytest.mark.skipif(not os.path.exists(LIB_PATH) or not os.path.exists(OBJDUMP), reason="needs the built library and llvm-objdump")
def test_wait_states_of_the_built_kernels(tmp_path):
    found, loads = [], 0
    for k, obj in enumerate(code_objects(LIB_PATH)):
        f = tmp_path / f"{k}.co"
        f.write_bytes(obj)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", str(f)], capture_output=True, text=True, check=True).stdout
        kernel, lines = None, []
        for raw in text.splitlines() + ["<end>:"]:
            m = re.match(r"(?:[0-9a-f]+ )?<(\S+)>:$", raw.strip())
            if m:
                found += [(kernel,) + v for v in violations(lines)]
                loads += sum("global_load_lds" in l for l in lines)
                kernel, lines = m[1], []
                continue
            t = raw.split("//")[0].strip()
            if t and not t.endswith(":"):
                lines.append(t)
    assert loads > 1000, "no loads to LDS found: the disassembly is not what this test reads"
    assert not found, f"{len(found)} places, among them {found[:3]}"

