"""What instructions written by hand owe the compiler and the hardware, read from the sources."""
import os
import re

from gpullama3_java_amd.csrc import build

BLOCK = re.compile(r'asm\s+(?:volatile)?\s*\((.*?)\);', re.S)


def blocks():
    for path in build.sources() + build.headers():
        with open(path) as f:
            text = f.read()
        for m in BLOCK.finditer(text):
            template, _, operands = m.group(1).partition(":")
            yield os.path.basename(path), template, operands


def test_m0_is_an_operand_where_an_instruction_uses_it():
    """A load into shared memory takes its address from m0. Set inside the block, the compiler would not know that the
    register has changed (it is a reserved one: a clobber of it is not honoured); as an operand the compiler sets it."""
    found = 0
    for where, template, operands in blocks():
        assert "m0" not in template, (where, template)
        if re.search(r"_load_\S+.*\blds\b", template):
            assert '"{m0}"' in operands, (where, template)
            found += 1
    assert found
