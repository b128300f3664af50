"""Wait states before the copies from global memory straight into LDS, in the built library's code.

The copies are written in inline assembly, which the compiler's hazard recogniser does not look into, and
M0, the LDS address, is read without an interlock: it needs one wait state after a scalar instruction has
written it (AMD Instinct MI300 instruction set architecture, "Manually inserted wait states"). Each
instruction between is one wait state and s_nop N is N + 1. The check reads the gfx950 code of the library
that was built here and walks back from every copy along every path."""
import os
import re
import subprocess

import pytest

from telmo_amd import build

OBJDUMP = os.environ.get("LLVM_OBJDUMP", "/opt/rocm/llvm/bin/llvm-objdump")
LINE = re.compile(r"^\t(?P<text>\S.*?)\s*// (?P<at>[0-9A-F]+):.*?(?:<(?P<sym>[^>+]+)\+0x(?P<off>[0-9a-f]+)>)?$")
SYMBOL = re.compile(r"^(?P<at>[0-9a-f]+) <(?P<name>.+)>:$")
COPY = re.compile(r"(global|buffer|scratch)_load_.*\blds\b|(global|scratch)_load_lds_")
STATES = 1  # the most that a write of an operand needs


def too_early(text, states, copy):
    """Whether `text`, `states` wait states before `copy`, writes an operand that needs more."""
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
