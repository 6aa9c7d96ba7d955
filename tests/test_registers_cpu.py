"""Registers that the built kernels spill: the figures the sources and documents state, from the library's own metadata."""
import re

from elmo_amd import _lib, build


def spilled():
    """{kernel: spilled vector registers} of the code objects in the library."""
    _lib.load()
    blob = open(build.OUT, "rb").read()
    found = {}
    # a kernel's entry is a MessagePack map with its keys in order, the count a small integer
    for name, count in re.findall(rb"\.name[^_]{1,2}(_ZN3xmc\w+).{1,400}?\.vgpr_spill_count([\x00-\x7f])", blob, re.S):
        found[name.decode()] = count[0]
    return found


def test_spilled_registers_are_those_stated():
    found = spilled()
    role = {tuple(map(int, re.search(r"ILi(\d)ELb(\d)ELi(\d)E", n).groups())): c for n, c in found.items() if "fp8_step_role_kernel" in n}
    one_pass = {n: c for n, c in found.items() if "cluster_step_kernel" in n}
    assert len(role) == 12 and len(one_pass) == 45
    assert set(one_pass.values()) == {0}
    for (mode, decay, head), count in role.items():       # mode 0 nearest, 1 Philox, 2 sr_fast; head: type of the compensation terms
        most = 8 if head else 4 if mode == 1 else 0
        assert count <= most, (mode, decay, head, count)
