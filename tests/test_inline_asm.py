"""What instructions written by hand owe the compiler and the hardware, read from the sources."""
import os
import re

from gpullama3_java_amd.csrc import build

BLOCK = re.compile(r'\basm\s*(?:volatile)?\s*\((.*?)\);', re.S)


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


def test_loads_by_hand_wait_for_their_scalar_operands():
    """A memory instruction may read a scalar register five wait states after a vector instruction wrote it; the compiler does not
    look into a block to keep them. So a block that loads copies its scalar offset by a scalar instruction first (whose result may
    be read at once), and the descriptor is put together by such instructions."""
    found = 0
    for where, template, operands in blocks():
        if re.search(r"(buffer|global|flat)_(load|store|atomic)", template):
            copied = re.match(r'"s_mov_b32 (%\d+), %\d+\\n\\tbuffer_load_dwordx4 (%\d+), (%\d+), (%\d+) offen lds"', template.strip())
            assert copied and copied.group(1) == copied.group(4) == "%0" and '"=&s"(' in operands, (where, template)
            with open(os.path.join(build.HERE, where)) as f:
                rsrc = re.search(r"i32x4 mf_rsrc\(.*?\n}", f.read(), re.S).group(0)
            assert rsrc.count('asm("s_mov_b32 %0, %1"') == rsrc.count("readfirstlane") == 2
            found += 1
    assert found


def test_no_vector_instruction_is_written_by_hand():
    """A vector instruction may read a matrix instruction's result only some wait states after it; the compiler keeps them for its own
    instructions and does not look into a block."""
    for where, template, operands in blocks():
        assert not re.search(r"\bv_\w+", template), (where, template)
