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


def registers(operand):
    """v0 .. and a0 .. of an operand, s0 .. and vcc as numbers (vcc: 106 and 107)."""
    operand = operand.strip("-|")
    m = re.fullmatch(r"([va])\[(\d+):(\d+)\]", operand)
    if m:
        return {m[1] + str(i) for i in range(int(m[2]), int(m[3]) + 1)}
    return {operand} if re.fullmatch(r"[va]\d+", operand) else {106, 107} if operand == "vcc" else scalars(operand)


def results(op, ops):
    """The operands that a vector instruction writes: the first, and of those with a carry or flag the second."""
    return ops[:2] if re.search(r"_co_|div_scale|mad_[ui]64", op) else ops[:1]


def union(operands):
    return set().union(*map(registers, operands))


def operands(line):
    rest = line.split(None, 1)
    return [o.strip().split()[0] for o in rest[1].split(",")] if len(rest) > 1 else []


def violations(lines):
    """(what, wait states between, instruction before, instruction) of straight-line code.  A vector instruction's write of a scalar register and a
    vector memory instruction that reads it: 5, a vector instruction that reads it: 2, unless a scalar instruction that uses the register, and waits
    for it, stands between; of a vector or accumulation register and a matrix instruction that reads it: 2; a write of M0 and a load to LDS: 1."""
    out = []
    for i, line in enumerate(lines):
        op, ops = line.split()[0], operands(line)
        memory, vector = re.match(r"(global|buffer|flat|scratch)_(load|store|atomic)", line), op.startswith("v_")
        if not memory and not vector:
            continue
        read = union(ops) if memory else union(ops[len(results(op, ops)):])
        reads, operand_reads = {r for r in read if isinstance(r, int)}, {r for r in read if op.startswith("v_mfma") and isinstance(r, str)}
        needed = 5 if memory else 2
        to_lds = memory and ("_lds_" in line or line.endswith(" lds"))
        waits = 0
        for before in reversed(lines[max(i - needed, 0):i]):
            bop, bops = before.split()[0], operands(before)
            written = union(results(bop, bops)) if bop.startswith("v_") else set()
            if written & reads:
                out.append(("scalar register", waits, before, line))
            if written & operand_reads and not bop.startswith("v_mfma"):
                out.append(("operand of a matrix instruction", waits, before, line))
            if to_lds and waits < 1 and bops[:1] == ["m0"]:
                out.append(("M0", waits, before, line))
            if bop in ("s_branch", "s_endpgm", "s_setpc_b64"):   # nothing falls through
                break
            if bop.startswith("s_"):
                reads -= union(bops)
            waits += int(bops[0], 0) + 1 if bop == "s_nop" else 1
            if waits >= needed:
                break
    return out


def overwritten(lines):
    """(wait states between, matrix instruction, instruction): a vector instruction that writes the vector registers of a matrix instruction's C operand
    while it may still read them, within 3 wait states of one of four passes (16x16x32) or 7 of one of eight (32x32x16).  Such an instruction takes its
    passes before the next one of its kind can start."""
    out = []
    for i, line in enumerate(lines):
        if not line.startswith("v_mfma"):
            continue
        ops = operands(line)
        c = {r for r in registers(ops[3]) - registers(ops[0]) if str(r).startswith("v")}
        needed, waits = (7 if "32x32" in line else 3), 0
        for after in lines[i + 1:i + 1 + needed] if c else []:
            op, after_ops = after.split()[0], operands(after)
            if op.startswith("v_") and not op.startswith("v_mfma") and union(results(op, after_ops)) & c:
                out.append((waits, line, after))
            if op in ("s_branch", "s_endpgm", "s_setpc_b64"):
                break
            waits += int(after_ops[0], 0) + 1 if op == "s_nop" else (8 if "32x32" in op else 4) if op.startswith("v_mfma") else 1
            if waits >= needed:
                break
    return out


def too_early(lines, targets=()):
    """(wait states between, matrix instruction, instruction): an instruction that reads or overwrites what a matrix instruction writes before it is
    there: within 8 wait states of one of four passes (16x16x32), 12 of one of eight (32x32x16).  A matrix instruction begins when the one before it has
    taken its passes, whatever stands between the two; it takes a result over by itself as C operand in the same registers, and writes behind the one
    before it.  `targets`: where
    branches lead ({line: line}); both ways are followed."""
    targets, out = dict(targets), []

    def passes(line):
        return 8 if "32x32" in line else 4

    for i, start in enumerate(lines):
        if not start.startswith("v_mfma"):
            continue
        result = registers(operands(start)[0])
        needed = passes(start) + 4
        todo, seen = [(i + 1, 0, passes(start))], set()   # line, wait states so far, wait states from which a matrix instruction can begin
        while todo:
            at, waits, free = todo.pop()
            if at >= len(lines) or (at, waits, free) in seen:
                continue
            seen.add((at, waits, free))
            op, ops = lines[at].split()[0], operands(lines[at])
            product = op.startswith("v_mfma")
            if product:
                waits = max(waits, free - 1)
            if waits >= needed:
                continue
            touched = union(ops[1:3] if product and registers(ops[3]) == result else ops[1:] if product else ops)
            if touched & result and re.match(r"v_|ds_|global_|scratch_|buffer_|flat_", op):
                out.append((waits, start, lines[at]))
                continue
            if product:
                free = waits + 1 + passes(lines[at])
            after = waits + (int(ops[0], 0) + 1 if op == "s_nop" else 1)
            if op not in ("s_branch", "s_endpgm", "s_setpc_b64"):
                todo.append((at + 1, after, free))
            if at in targets:
                todo.append((targets[at], after, free))
    return out


def in_flight(lines):
    """(read of LDS, instruction): an instruction that touches the registers of an LDS read ahead of a wait for it, in straight-line code.  Reads come back
    in their order, so that a later one may bring the same registers."""
    out = []
    for i, read in enumerate(lines):
        if not read.startswith("ds_read"):
            continue
        result, behind = registers(operands(read)[0]), 0
        for after in lines[i + 1:]:
            op, ops = after.split()[0], operands(after)
            m = re.search(r"lgkmcnt\((\d+)\)", after)
            if (m and int(m[1]) <= behind) or op in ("s_branch", "s_endpgm", "s_setpc_b64"):
                break
            if union(ops[1:] if op.startswith("ds_read") else ops) & result:
                out.append((read, after))
                break
            behind += bool(re.match("ds_|s_load|s_buffer_load", op))
    return out


def test_hazards_planted_in_a_listing_are_found():
    load = "global_load_lds_dwordx4 v1, s[0:1] offset:2048"
    assert violations(["v_readlane_b32 s1, v252, 18", load])
    assert violations(["v_readfirstlane_b32 s0, v2", "s_nop 1", "s_mov_b32 m0, s3", "s_nop 0", load])
    assert violations(["s_mov_b32 m0, s3", load]) and not violations(["s_mov_b32 m0, s3", "s_nop 0", load])
    assert not violations(["v_readfirstlane_b32 s0, v2", "s_nop 4", load])
    assert not violations(["v_readfirstlane_b32 s0, v2", "s_mov_b64 s[0:1], s[0:1]", load])
    assert not violations(["v_readfirstlane_b32 s2, v2", "s_mov_b32 m0, s3", "s_nop 0", load])

    select = "v_cndmask_b32_e64 v3, 0, -1, s[4:5]"
    assert violations(["v_readlane_b32 s5, v252, 18", select])
    assert violations(["v_cmp_gt_i32_e32 vcc, v1, v2", "v_mov_b32_e32 v9, v8", "v_cndmask_b32_e32 v3, 0, v4, vcc"])
    assert violations(["v_add_co_u32_e64 v1, s[4:5], v2, v3", "s_nop 0", select])
    assert violations(["v_readfirstlane_b32 s7, v2", "v_add_u32_e32 v3, s7, v4"])
    assert not violations(["v_readlane_b32 s5, v252, 18", "s_nop 1", select])
    assert not violations(["v_readlane_b32 s5, v252, 18", "s_mov_b64 s[4:5], s[4:5]", select])
    assert not violations(["s_mov_b32 s5, 0xff00ff00", select]) and not violations([select, "v_readlane_b32 s5, v252, 18"])

    product = "v_mfma_f32_32x32x16_bf16 v[0:15], v[16:19], a[20:23], v[0:15]"
    assert violations(["v_cvt_pk_bf16_f32 v19, v40, v41", "v_mov_b32_e32 v50, v51", product])
    assert violations(["v_accvgpr_write_b32 a20, v3", product]) and violations(["v_accvgpr_read_b32 v15, a3", "s_nop 0", product])
    assert not violations(["v_cvt_pk_bf16_f32 v19, v40, v41", "s_nop 1", product])
    assert not violations(["v_mov_b32_e32 v24, v40", product]) and not violations(["ds_read_b128 v[16:19], v60", product])

    start = "v_mfma_f32_16x16x32_bf16 v[78:81], v[104:107], a[32:35], v[10:13]"
    assert overwritten([start, "v_fma_f32 v11, v74, v128, -v189"]) and overwritten([start, "s_nop 1", "v_mov_b32_e32 v13, v1"])
    assert not overwritten([start, "s_nop 2", "v_mov_b32_e32 v13, v1"]) and not overwritten([start, "v_mov_b32_e32 v80, v10"])
    assert not overwritten([start, "v_mfma_f32_16x16x32_bf16 v[82:85], v[104:107], a[36:39], v[14:17]", "v_mov_b32_e32 v13, v1"])
    assert overwritten([start.replace("16x16x32", "32x32x16"), "s_nop 5", "v_mov_b32_e32 v13, v1"])

    other = "v_mfma_f32_16x16x32_bf16 v[82:85], v[104:107], a[36:39], v[14:17]"
    read, keep, store = "v_fma_f32 v1, v80, v2, v3", "ds_write_b64 v60, v[78:79]", "global_store_dwordx4 v[2:3], v[78:81], off"
    assert all(too_early([start, x]) and too_early([start, "s_nop 6", x]) and not too_early([start, "s_nop 7", x]) for x in (read, keep, store, "v_mov_b32_e32 v81, v1"))
    assert too_early([start, other, read]) and not too_early([start, other, other, read]) and not too_early([start, "v_mov_b32_e32 v9, v8"] * 8)
    assert too_early([start, "v_mov_b32_e32 v9, v8", "v_mov_b32_e32 v9, v8", other, "s_nop 2", read])   # (what stands ahead of the second is not counted twice)
    assert not too_early([start, "v_mov_b32_e32 v9, v8", "v_mov_b32_e32 v9, v8", other, "s_nop 3", read])
    assert too_early([start, "v_mfma_f32_16x16x32_bf16 v[82:85], v[78:81], a[36:39], v[14:17]"])         # as an operand
    assert too_early([start, "v_mfma_f32_16x16x32_bf16 v[82:85], v[104:107], a[36:39], v[80:83]"])       # as C, in part
    assert not too_early([start, "v_mfma_f32_16x16x32_bf16 v[78:81], v[104:107], a[36:39], v[78:81]"])   # summed up on top
    eight = start.replace("16x16x32", "32x32x16").replace("v[78:81]", "v[78:93]").replace("v[10:13]", "v[10:25]")
    assert too_early([eight, "s_nop 10", read]) and not too_early([eight, "s_nop 11", read])
    assert too_early([read, "s_nop 7", start, "s_cbranch_scc1 65533"], {3: 0}) and not too_early([read, "s_nop 7", start, "s_cbranch_scc1 65534"], {3: 1})

    read = "ds_read_b128 v[64:67], v62"
    assert in_flight([read, "v_cvt_pk_bf16_f32 v64, v77, v78"]) and in_flight([read, "ds_read_b128 v[68:71], v62", "s_waitcnt lgkmcnt(1)", "ds_write_b64 v1, v[66:67]"]) == []
    assert in_flight([read, "ds_read_b128 v[68:71], v62", "s_waitcnt lgkmcnt(1)", "v_mov_b32_e32 v1, v70"]) and not in_flight([read, read, "s_waitcnt lgkmcnt(0)", "v_mov_b32_e32 v1, v64"])


@pytest.fixture(scope="module")
def listings(tmp_path_factory):
    """(kernel, its instructions, {branch: where it leads}) of every kernel of the library, both places as indexes of instructions."""
    if not os.path.exists(OBJDUMP):
        pytest.skip("needs llvm-objdump")
    assert os.path.exists(LIB_PATH), "the library is not built"
    out = []
    for k, obj in enumerate(code_objects(LIB_PATH)):
        f = tmp_path_factory.mktemp("code") / f"{k}.co"
        f.write_bytes(obj)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(f)], capture_output=True, text=True, check=True).stdout
        for part in re.split(r"^[0-9a-f]+ <(?=\S+>:$)", text, flags=re.M)[1:]:
            lines, places, leads = [], {}, {}
            for t, place in re.findall(r"^\s+(\S.*?)\s*// ([0-9A-F]+):", part, flags=re.M):
                places[int(place, 16)] = len(lines)
                m = re.match(r"s_c?branch\S* (\d+)", t)
                if m:   # (a signed number of words from the next instruction on)
                    leads[len(lines)] = int(place, 16) + 4 + 4 * ((int(m[1]) ^ 0x8000) - 0x8000)
                lines.append(t)
            out.append((part[:part.index(">")], lines, {at: places[to] for at, to in leads.items() if to in places}))
    return out


def test_wait_states_of_the_built_kernels(listings):
    found, loads, products = [], 0, 0
    for kernel, lines, leads in listings:
        found += [(kernel,) + v for v in violations(lines) + overwritten(lines) + too_early(lines, leads) + in_flight(lines)]
        loads += sum("global_load_lds" in l for l in lines)
        products += sum(l.startswith("v_mfma") for l in lines)
    assert loads > 1000 and products > 1000, "no loads to LDS, no matrix instructions: the disassembly is not what this test reads"
    assert not found, f"{len(found)} places, among them {found[:3]}"


def test_block_loops_of_the_backward_kernels_reload_nothing(listings):
    """No register parked in scratch memory comes back inside the loops over blocks or tiles: the wait for it is a wait for every load to LDS on its
    way.  A loop is what lies between a branch back and where it leads; the body of a block has 64 or 128 matrix instructions, a round of four 512, and
    the loops around those loops, over tasks and items, have more."""
    loops, found = 0, []
    for kernel, lines, leads in listings:
        for at, to in leads.items() if "ca_bwd" in kernel else ():
            body = lines[to:at + 1]
            if any("global_load_lds" in l for l in body) and sum(l.startswith("v_mfma") for l in body) <= 512:
                loops += 1
                found += [(kernel, len(body), l) for l in body if l.startswith("scratch_load")]
    assert loops > 100, "the disassembly is not what this test reads"
    assert not found, f"{len(found)} reloads, among them {found[:3]}"
