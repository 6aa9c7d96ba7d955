"""Registers that the built kernels spill: the figures the sources and documents state, from the library's own metadata."""
import re

from elmo_amd import _lib, build


def spilled():
    """{kernel: spilled vector registers} of the code objects in the library."""
    _lib.load()
    blob = open(build.OUT, "rb").read()
    # a kernel's entry is a MessagePack map with its keys in order; the count takes one byte, or up to four behind a type byte
    found = re.findall(rb"\.name[^_]{1,2}(_ZN3xmc\w+|_Z\w+).{1,400}?\.vgpr_spill_count([\x00-\x7f]|\xcc.|\xcd..|\xce....)", blob, re.S)
    assert len(found) == len(re.findall(rb"\.vgpr_spill_count", blob)), "an entry that this does not understand"
    names = [name.decode() for name, _ in found]
    assert len(set(names)) == len(names)
    return {name: int.from_bytes(count[1:] or count, "big") for name, (_, count) in zip(names, found)}


def test_spilled_registers_are_those_stated():
    found = spilled()
    # all of a kernel's variants, by all that they differ in (template arguments)
    role = {tuple(map(int, re.search(r"ILi(\d)ELb(\d)ELi(\d)ELi(\d)EEE", n).groups())): c for n, c in found.items() if "fp8_step_role_kernel" in n}
    one_pass = {tuple(map(int, re.search(r"ILi(\d)ELi(\d)ELi(\d)ELi(\d)ELi(\d)EEE", n).groups())): c for n, c in found.items() if "cluster_step" in n}
    assert set(role) == ({(mode, 0, 0, blocks) for mode in range(3) for blocks in (1, 2, 3, 4)} | {(mode, 1, 0, 4) for mode in range(3)} |
                         {(mode, 0, head, blocks) for mode in range(3) for head in (1, 2) for blocks in (2, 4)})
    assert set(one_pass) == {(weights, fp8, members, blocks, mode) for weights, fp8 in ((0, 0), (0, 1), (1, 0)) for mode in range(3)
                             for members, blocks in ((1, 2), (1, 4), (2, 4), (3, 4), (4, 4), (6, 4), (8, 4))}
    assert set(one_pass.values()) == {0}
    for (mode, decay, head, blocks), count in role.items():       # mode 0 nearest, 1 Philox, 2 sr_fast; head: type of the compensation terms
        most = 0 if blocks < 4 else 8 if head else 3 if mode == 1 else 0
        assert count <= most, (mode, decay, head, blocks, count)
