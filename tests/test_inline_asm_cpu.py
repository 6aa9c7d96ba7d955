"""Hardware hazards inside inline assembly, which the compiler does not look into."""
import glob
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MEMORY = r"(global|flat|buffer|scratch)_(load|store|atomic)"


def states(lines):
    """Wait states that these instructions are: one each, s_nop N counts N + 1."""
    return sum(int(l.split()[1]) + 1 if l.startswith("s_nop") else 1 for l in lines)


def hazards(source):
    """(faults, memory instructions seen) of every asm statement of a source.  The wait states of gfx950, as hipcc itself keeps them
    around the same instructions that it generates: five between a vector instruction that writes a scalar register (v_readlane
    of a spilled scalar, v_readfirstlane) and a memory instruction that has it as its address; one between a write of M0 and a load
    into LDS; two between a store of more than 8 bytes and a vector instruction that overwrites the registers it reads.  What stands in
    front of the statement and behind it is the compiler's choice, so all of them have to be inside."""
    faults, seen = [], 0
    for text, rest in re.findall(r'asm volatile\(((?:\s*"(?:[^"\\]|\\.)*")+)([^;]*);', source):
        constraints = re.findall(r'"[=+&]*([a-z])"\s*\(', rest)
        lines = [l.strip() for part in re.findall(r'"((?:[^"\\]|\\.)*)"', text) for l in part.replace("\\t", " ").split("\\n")]
        for i, line in enumerate(lines):
            if not re.match(MEMORY, line):
                continue
            seen += 1
            operands = [constraints[int(n)] for n in re.findall(r"%(\d+)", line)]
            if "s" in operands and states(lines[:i]) < 5:
                faults.append(("scalar address", line))
            if "_load_lds_" in line:
                m0 = [k for k in range(i) if re.match(r"s_\w+ m0,", lines[k])]
                if not m0 or states(lines[m0[-1] + 1:i]) < 1:
                    faults.append(("M0", line))
            if re.search(r"_store_dwordx[34]\b", line):
                behind = [l for l in lines[i + 1:i + 2] if l.startswith("s_nop")]
                if states(behind) < 2:
                    faults.append(("wide store", line))
    return faults, seen


def test_inline_assembly_brings_its_own_wait_states():
    total = 0
    for path in glob.glob(os.path.join(ROOT, "elmo_amd", "csrc", "*")):
        source = open(path).read()
        faults, seen = hazards(source)
        assert not faults, (os.path.basename(path), faults)
        assert seen == len(re.findall(MEMORY + r"_\w+ %\d", source)), os.path.basename(path)     # (none escaped the parser)
        total += seen
    assert total > 0


@pytest.mark.parametrize("body,operands,fault", [
    (r"s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2", '"s"(l), "v"(o), "s"(b)', "scalar address"),
    (r"s_mov_b32 m0, %0\n\ts_nop 2\n\tglobal_load_lds_dwordx4 %1, %2", '"s"(l), "v"(o), "s"(b)', "scalar address"),
    (r"s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2", '"s"(l), "v"(o), "s"(b)', None),
    (r"s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, off", '"s"(l), "v"(g)', "M0"),
    (r"s_nop 4\n\ts_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2", '"s"(l), "v"(o), "s"(b)', "M0"),
    (r"s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off", '"s"(l), "v"(g)', None),
    (r"s_nop 3\n\tglobal_store_dwordx2 %0, %1, %2", '"v"(a), "v"(d), "s"(b)', "scalar address"),
    (r"s_nop 4\n\tglobal_store_dwordx2 %0, %1, %2", '"v"(a), "v"(d), "s"(b)', None),
    (r"global_store_dwordx4 %0, %1, off", '"v"(a), "v"(d)', "wide store"),
    (r"global_store_dwordx3 %0, %1, off\n\ts_nop 0", '"v"(a), "v"(d)', "wide store"),
    (r"global_store_dwordx4 %0, %1, off\n\ts_waitcnt vmcnt(0)\n\ts_nop 1", '"v"(a), "v"(d)', "wide store"),
    (r"global_store_dwordx4 %0, %1, off\n\ts_nop 1", '"v"(a), "v"(d)', None),
])
def test_missing_wait_states_are_found(body, operands, fault):
    faults, seen = hazards('  asm volatile("%s" : : %s : "memory", "m0");' % (body, operands))
    assert seen == 1 and [f[0] for f in faults] == ([fault] if fault else [])
