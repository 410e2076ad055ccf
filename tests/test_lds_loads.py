"""Loads from memory straight into LDS, written out as inline assembly: what the compiler cannot check in them."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mimir_amd", "csrc")


def statements():
    for path in sorted(glob.glob(os.path.join(CSRC, "*"))):
        if os.path.isfile(path):
            with open(path) as f:
                for n, line in enumerate(f, 1):
                    for text in re.findall(r'\basm\s+(?:volatile\s*)?\(\s*"((?:[^"\\]|\\.)*)"', line):
                        yield pytest.param([i.strip() for i in text.replace("\\t", "").split("\\n")], id=f"{os.path.basename(path)}:{n}")


@pytest.mark.parametrize("instructions", [p for p in statements() if any("_lds_" in i or re.search(r"\blds\b|\bm0\b", i) for i in p.values[0])])
def test_a_wait_state_lies_between_m0_and_the_load_that_reads_it(instructions):
    """gfx9: a load into LDS takes its base from M0 and may not come right behind a scalar write of it (one wait state); the
    statement sets M0 itself, since the compiler does not know that the load reads it."""
    assert [i.split()[0] for i in instructions[:2]] == ["s_mov_b32", "s_nop"] and instructions[0].split()[1] == "m0,"
    assert len(instructions) == 3 and "_lds_" in instructions[2]
