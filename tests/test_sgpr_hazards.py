"""A vector memory instruction may read a scalar register only five wait states after a vector instruction (a
v_readfirstlane, a v_readlane of a spilled scalar, a compare) has written it, and an LDS copy M0 only one after it was written.
The compiler pads its own instructions and looks into no assembly statement, so the built library is read back: every kernel, every
path into every vector memory instruction."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "kernels_amd", "streaming_attention", "libstreaming_attention.so")
OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
VMEM = ("buffer_", "global_", "flat_", "scratch_")
VALU_TO_VMEM, M0_TO_LDS_COPY = 5, 1


def scalars(operand):
    """The scalar registers that an operand names, as numbers, or 'vcc' / 'm0'."""
    out = set()
    for m in re.finditer(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b|\b(vcc|m0)\b", operand):
        if m.group(4):
            out.add(m.group(4))
        elif m.group(3):
            out.add(int(m.group(3)))
        else:
            out.update(range(int(m.group(1)), int(m.group(2)) + 1))
    return out


def parse(text):
    """([(mnemonic, operands, wait states, line, last label)], predecessors) of an object's disassembly."""
    code, at, jumps, label = [], {}, [], ""
    for line in text.splitlines():
        label = line.split("<")[-1].rstrip(">:") if re.match(r"[0-9a-f]+ <", line) else label
        m = re.match(r"\s+(\w+)\s*(.*?)\s*// ([0-9A-F]+): ([0-9A-F]+)", line)
        if not m:
            continue
        op, args, addr = m.group(1), m.group(2), int(m.group(3), 16)
        at[addr] = len(code)
        if op.startswith(("s_branch", "s_cbranch")):
            offset = int(m.group(4)[-4:], 16)   # of the encoding: the text may name a label
            jumps.append((len(code), addr + 4 + 4 * (offset - 65536 if offset > 32767 else offset)))
        states = int(args.split()[0], 0) + 1 if op == "s_nop" else 1
        code.append((op, [a.strip() for a in args.split(",")], states, line.split("//")[0].strip(), label))
    before = [[i - 1] if i and code[i - 1][0] not in ("s_branch", "s_endpgm", "s_setpc_b64") else [] for i in range(len(code))]
    for source, target in jumps:
        before[at[target]].append(source)
    return code, before


def written_by_valu(op, args):
    if not op.startswith("v_"):
        return set()
    out = scalars(args[0])
    if "_co_" in op or op.startswith("v_div_scale"):   # the carry is the second result
        out |= scalars(args[1])
    return out


def hazards(code, before):
    found = []
    for i, (op, args, _, line, label) in enumerate(code):
        if not op.startswith(VMEM):
            continue
        reads = set().union(*(scalars(a) for a in args))
        lds_copy = re.search(r"\blds\b", line) is not None or "_lds_" in op
        todo, seen = [(p, 0) for p in before[i]], set()
        while todo:
            j, states = todo.pop()   # `states` wait states lie between instruction j and the memory instruction
            if states >= VALU_TO_VMEM or (j, states) in seen:
                continue
            seen.add((j, states))
            o, a, n, text, _ = code[j]
            if written_by_valu(o, a) & reads:
                found.append(f"{label}: {text} .. {states} wait states .. {line}")
                continue
            if lds_copy and states < M0_TO_LDS_COPY and o.startswith("s_") and scalars(a[0]) == {"m0"}:
                found.append(f"{label}: {text} .. {states} wait states .. {line}")
            todo += [(p, states + n) for p in before[j]]
    return found


def test_scan_finds_what_it_looks_for():
    """Planted in a listing: two short of the five wait states, reached over a branch, M0 right before a copy; and none where padded."""
    def one(*lines):
        return parse("".join(f"\t{t}  // {4 * i:012X}: BF820001\n" for i, t in enumerate(lines)))

    load = "buffer_load_dwordx4 v0, s[4:7], s9 offen lds"
    assert len(hazards(*one("v_readfirstlane_b32 s6, v1", "s_mov_b32 m0, s3", "s_nop 0", load))) == 1
    assert len(hazards(*one("v_readlane_b32 s9, v1, 3", "s_mov_b32 m0, s3", "s_nop 2", load))) == 1
    assert len(hazards(*one("v_cmp_lt_i32_e64 s[8:9], v0, v1", "s_branch 1", "s_endpgm", "s_mov_b32 m0, s3", "s_nop 0", load))) == 1
    assert len(hazards(*one("s_mov_b32 m0, s3", load))) == 1
    assert hazards(*one("v_readfirstlane_b32 s6, v1", "s_mov_b32 m0, s3", "s_nop 3", load)) == []
    assert hazards(*one("v_readfirstlane_b32 s3, v1", "s_mov_b32 m0, s3", "s_nop 0", load)) == []


@pytest.mark.skipif(not (os.path.exists(LIB) and os.path.exists(OBJDUMP)), reason="no built library or no disassembler")
def test_no_kernel_reads_a_scalar_too_early(tmp_path):
    shutil.copy(LIB, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    objects = sorted(f for f in os.listdir(tmp_path) if "gfx950" in f)
    assert objects
    found, copies = [], 0
    for f in objects:
        listing = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", f], cwd=tmp_path, check=True, capture_output=True, text=True).stdout
        code, before = parse(listing)
        copies += sum(line.endswith(" lds") for _, _, _, line, _ in code)
        found += hazards(code, before)
    assert copies > 500   # the listing was understood
    assert not found, "\n".join(found)
