"""Hardware hazards inside inline assembly, which the compiler does not look into."""
import glob
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_inline_assembly_brings_its_own_wait_states():
    """gfx9: a vector instruction right behind a store of more than 8 bytes may overwrite the registers the store still reads, and
    a load into LDS right behind a write of M0 may still see the old value (one wait state each).  The compiler inserts these
    around its own instructions only."""
    wide = loads = 0
    for path in glob.glob(os.path.join(ROOT, "elmo_amd", "csrc", "*")):
        text = open(path).read()
        for text_of_asm in re.findall(r'asm volatile\(((?:\s*"(?:[^"\\]|\\.)*")+)', text):
            lines = [l.strip() for part in re.findall(r'"((?:[^"\\]|\\.)*)"', text_of_asm) for l in part.replace("\\t", " ").split("\\n")]
            for i, line in enumerate(lines):
                if re.match(r"(global|flat|buffer|scratch)_store_dwordx[34]\b", line):
                    wide += 1
                    assert i + 1 < len(lines) and re.match(r"s_nop [0-9]+$", lines[i + 1]), (os.path.basename(path), line)
                if "_load_lds_" in line:
                    loads += 1
                    assert i > 0 and re.match(r"s_nop [0-9]+$", lines[i - 1]), (os.path.basename(path), line)
    assert wide > 0 and loads > 0
