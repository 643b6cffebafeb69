"""What can be said of the kernels' sources without a GPU."""
import os
import re

import pytest

from infinilm_amd.csrc import build


def _statements(text, word):
    """The arguments of every `word(...)` in a source."""
    for m in re.finditer(r"\b%s\s*\(" % word, text):
        depth, i = 1, m.end()
        while depth:
            depth += {"(": 1, ")": -1}.get(text[i], 0)
            i += 1
        yield text[m.end():i - 1]


@pytest.mark.parametrize("name", build.sources())
def test_assembly_names_the_registers_it_writes(name):
    """m0 written in an asm statement is named as clobbered: the compiler may hold a value of its own there."""
    with open(os.path.join(build.HERE, name)) as f:
        text = f.read()
    for word in ("asm volatile", "asm"):
        for s in _statements(text, word):
            if re.search(r"\bm0\s*,", s):
                assert '"m0"' in s, s
