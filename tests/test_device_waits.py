"""Wait states before the copies from global memory straight into LDS, in the built library's code.

The copies are written in inline assembly, which the compiler's hazard recogniser does not look into, and
two of their operands are read without an interlock (AMD Instinct MI300 instruction set architecture,
"Manually inserted wait states"): M0, the LDS address, needs one wait state after a scalar instruction has
written it, and the scalar registers of the global address need five after a vector instruction (a
v_readfirstlane_b32, or the v_readlane_b32 of a spilled register) has. Each instruction between is one
wait state and s_nop N is N + 1. The check reads the gfx950 code of the library that was built here and
walks back from every copy along every path."""
import os
import re
import subprocess

import pytest

from telmo_amd import build

OBJDUMP = os.environ.get("LLVM_OBJDUMP", "/opt/rocm/llvm/bin/llvm-objdump")
LINE = re.compile(r"^\t(?P<text>\S.*?)\s*// (?P<at>[0-9A-F]+):.*?(?:<(?P<sym>[^>+]+)\+0x(?P<off>[0-9a-f]+)>)?$")
SYMBOL = re.compile(r"^(?P<at>[0-9a-f]+) <(?P<name>.+)>:$")
COPY = re.compile(r"(global|buffer|scratch)_load_.*\blds\b|(global|scratch)_load_lds_")
STATES = 5  # the most that a write of an operand needs


def sgprs(text):
    """The scalar registers that an operand text names, vcc as "vcc"."""
    found = set(re.findall(r"\bvcc\b", text))
    found.update(int(n) for n in re.findall(r"\bs(\d+)\b", text))
    for lo, hi in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        found.update(range(int(lo), int(hi) + 1))
    return found


def written(text):
    """The scalar registers that a vector instruction writes (its scalar destination operands)."""
    name, _, rest = text.partition(" ")
    operands = re.findall(r"[^\s,\[]+(?:\[[^\]]*\])?", rest)
    found = sgprs(operands[0]) if operands else set()
    # The carry-outs and div_scale's flag are second destinations.
    if re.match(r"v_(add|sub|subrev|addc|subb|subbrev)_co_u32|v_div_scale|v_mad_[iu]64", name) and len(operands) > 1:
        found |= sgprs(operands[1])
    return found


def too_early(text, states, copy):
    """Whether `text`, `states` wait states before `copy`, writes an operand that needs more."""
    if text.startswith("v_"):
        return states < 5 and bool(written(text) & sgprs(copy))
    return states < 1 and re.match(r"s_\S+ m0,", text) is not None


def hazards(lines):
    """([(address, copy, writer) of each copy that a write of its operands reaches too early], copies)."""
    code, index, symbols, targets = [], {}, {}, {}
    for line in lines:
        s = SYMBOL.match(line)
        if s:
            symbols[s["name"]] = int(s["at"], 16)
            continue
        i = LINE.match(line)
        if i:
            index[int(i["at"], 16)] = len(code)
            code.append((int(i["at"], 16), i["text"], i["sym"] and (i["sym"], int(i["off"], 16))))
    for n, (_, text, target) in enumerate(code):
        if text.startswith(("s_branch", "s_cbranch")) and target:
            targets.setdefault(index[symbols[target[0]] + target[1]], []).append(n)

    def before(n):  # the instructions that may run right before instruction n
        if n and not code[n - 1][1].startswith(("s_branch", "s_endpgm", "s_setpc_b64")):
            yield n - 1
        yield from targets.get(n, ())

    found, copies = [], 0
    for n, (at, copy, _) in enumerate(code):
        if not COPY.match(copy):
            continue
        copies += 1
        reached, todo = {}, [(p, 0) for p in before(n)]
        while todo:
            p, states = todo.pop()
            if states >= STATES or reached.get(p, STATES) <= states:
                continue
            reached[p] = states
            text = code[p][1]
            if too_early(text, states, copy):
                found.append((hex(at), copy, text))
            nop = re.match(r"s_nop (\d+)", text)
            todo += [(q, states + (int(nop[1]) + 1 if nop else 1)) for q in before(p)]
    return found, copies


def dump(*texts):
    return ["0000000000001000 <kernel>:"] + [f"\t{t}  // {0x1000 + 4 * i:012X}: 00000000" for i, t in enumerate(texts)]


def test_the_check_finds_an_early_lds_address():
    copy = "global_load_lds_dwordx4 v4, s[30:31]"
    assert hazards(dump("s_mov_b32 m0, s5", copy))[0]
    assert not hazards(dump("s_mov_b32 m0, s5", "s_nop 0", copy))[0]
    loop = dump("s_nop 0", copy, "s_add_u32 m0, s5, s6", "s_cbranch_scc1 65533")
    assert not hazards(loop)[0]  # the branch itself is a wait state
    loop = dump("s_nop 0", "s_nop 0", copy, "s_branch 65533")
    loop[-1] += " <kernel+0x8>"
    assert not hazards(loop)[0]


def test_the_check_finds_an_early_base():
    copy = "global_load_lds_dwordx4 v4, s[30:31]"
    assert hazards(dump("v_readfirstlane_b32 s31, v2", "s_mov_b32 m0, s5", "s_nop 2", copy))[0]
    assert not hazards(dump("v_readfirstlane_b32 s31, v2", "s_mov_b32 m0, s5", "s_nop 3", copy))[0]
    assert not hazards(dump("v_readfirstlane_b32 s32, v2", "s_mov_b32 m0, s5", "s_nop 0", copy))[0]
    assert hazards(dump("v_add_co_u32_e64 v1, s[30:31], v2, v3", "s_mov_b32 m0, s5", "s_nop 0", copy))[0]
    loop = dump("s_nop 0", "s_nop 0", copy, "v_cmp_lt_i32_e64 s[30:31], v2, v3", "s_cbranch_scc1 65532")
    loop[-1] += " <kernel+0x4>"
    assert hazards(loop)[0]


def test_copies_into_lds_wait_for_their_operands(tmp_path):
    if not os.path.exists(build.LIB):
        build.build()
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    lib = tmp_path / "lib.so"
    lib.symlink_to(build.LIB)
    subprocess.run([OBJDUMP, "--offloading", str(lib)], cwd=tmp_path, check=True, capture_output=True)
    total = 0
    for obj in sorted(tmp_path.glob("*gfx950")):
        code = subprocess.run([OBJDUMP, "-d", str(obj)], check=True, capture_output=True, text=True).stdout
        found, copies = hazards(code.splitlines())
        assert not found, (obj.name, len(found), copies, found[:8])
        total += copies
    assert total > 0, "no copies found: has the disassembly's form changed?"
