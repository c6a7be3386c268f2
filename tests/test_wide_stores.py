"""The 16-byte buffer stores of the built library against a gfx950 hazard, read from its assembly (CPU).

A store of more than 8 bytes needs two wait states before a vector instruction rewrites its data
registers. The compiler keeps them, except where the store's scalar offset is a register: there it
assumes that none are needed, and on gfx950 the store's first dword was then the new value in some
lanes, now and then. So every such store has to have two wait states behind it.
"""
import os
import re
import struct
import subprocess

import pytest

from ancha_amd import _native

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
WAIT_STATES = 2


def code_objects(path):
    """The gfx950 code objects of a library (clang's offload bundles, one per source file)."""
    data = open(path, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        entry = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            name = data[entry + 24:entry + 24 + length].decode()
            entry += 24 + length
            if "gfx950" in name and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + len(MAGIC))


def registers(operand):
    """The vector registers (v or a) that an operand names."""
    m = re.fullmatch(r"([va])\[(\d+):(\d+)\]", operand)
    if m:
        return {(m[1], i) for i in range(int(m[2]), int(m[3]) + 1)}
    m = re.fullmatch(r"([va])(\d+)", operand)
    return {(m[1], int(m[2]))} if m else set()


def operands(line):
    parts = line.split(None, 1)
    return [o.split()[0] for o in parts[1].split(",")] if len(parts) > 1 else []


def written(line):
    """The vector registers that a vector ALU (or matrix) instruction writes."""
    if not line.startswith("v_"):
        return set()
    return set().union(*(registers(o) for o in operands(line)[:2 if "swap" in line else 1]))


def short_gaps(lines):
    """(stores with a scalar offset register, those of them that lack the wait states). A branch
    inside them counts as lacking them: what follows is then not known from the listing's order."""
    stores, short = 0, []
    for i, line in enumerate(lines):
        if not re.match(r"buffer_store_dwordx[34] ", line):
            continue
        ops = operands(line)  # data, address, descriptor, scalar offset
        if not re.match(r"[a-z]", ops[3]):
            continue
        stores += 1
        states = 0
        for after in lines[i + 1:]:
            if states >= WAIT_STATES or after.startswith("s_endpgm"):
                break
            if after.startswith("s_nop"):
                states += int(operands(after)[0], 0) + 1
                continue
            if after.startswith(("s_cbranch", "s_branch", "s_setpc", "s_swappc")) or \
                    written(after) & registers(ops[0]):
                short.append(f"{line}  ->  {after}")
                break
            states += 1
    return stores, short


def test_rule_on_written_out_cases():
    store = "buffer_store_dwordx4 v[4:7], v1, s[0:3], s9 offen nt"
    for lines, bad in [
        ([store, "s_nop 0", "v_mov_b32_e32 v4, v0"], 1),
        ([store, "s_nop 1", "v_mov_b32_e32 v4, v0"], 0),
        ([store, "s_add_i32 s4, s4, 1", "v_add_u32_e32 v7, v0, v1"], 1),
        ([store, "s_nop 0", "v_mov_b32_e32 v8, v4", "v_mov_b32_e32 v4, v0"], 0),
        ([store, "v_mfma_f32_32x32x16_f16 a[0:15], v[4:7], v[8:11], a[0:15]", "s_nop 0"], 0),
        ([store, "v_swap_b32 v0, v6"], 1),
        ([store, "s_cbranch_scc1 12"], 1),
        ([store, "s_endpgm"], 0),
        ([store.replace("s9", "0"), "v_mov_b32_e32 v4, v0"], 0),  # the compiler's own case
    ]:
        assert len(short_gaps(lines)[1]) == bad, lines


def test_library_keeps_the_wait_states():
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump to read the assembly with")
    path = _native.lib()._name
    found, wide, short = 0, 0, []
    for i, code in enumerate(code_objects(path)):
        r = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", "--no-show-raw-insn",
                            "--no-leading-addr", "-"], input=code, capture_output=True, check=True)
        name, lines = f"code object {i}", []
        for text in r.stdout.decode().splitlines() + ["<end>:"]:
            label = re.match(r"(?:[0-9a-f]+ )?<(.*)>:$", text.strip())
            if label:
                stores, bad = short_gaps(lines)
                wide += stores
                short += [f"{name}: {b}" for b in bad]
                name, lines = label[1], []
            else:
                line = text.split("//")[0].strip()
                if line and text[:1].isspace():
                    lines.append(line)
        found += 1
    print(f"{found} code objects, {wide} wide stores with a scalar offset register")
    assert found > 1
    assert not short, "\n".join(short)
