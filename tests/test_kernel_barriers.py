"""The sources of the encoder kernels: a barrier stands in no branch that the blocks or lanes of a workgroup may take
differently (only in `if constexpr`, and in loops over what the whole workgroup shares)."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "s2tc_amd", "csrc")


def _enclosing(text):
    """The headers of the blocks around every __syncthreads()."""
    text = re.sub(r"//[^\n]*|/\*.*?\*/", "", text, flags=re.S)
    text = re.sub(r"^#(?:[^\n]*\\\n)*[^\n]*", "", text, flags=re.M)
    stack, head, at = [], "", 0
    for m in re.finditer(r"[{};]|__syncthreads\(\)", text):
        head += text[at:m.start()]
        at = m.end()
        if m.group() == "{":
            stack.append(head.strip())
            head = ""
        elif m.group() == "}":
            stack.pop()
            head = ""
        elif m.group() == ";":
            head = "" if head.count("(") == head.count(")") else head + ";"
        else:
            yield stack + [head.strip()]


@pytest.mark.parametrize("name", ["encode_normal.h", "kernels_cd.hip"])
def test_barriers_outside_branches(name):
    found = list(_enclosing(open(os.path.join(CSRC, name)).read()))
    assert found
    for blocks in found:
        for b in blocks:
            assert not re.search(r"(^|\s)(if(?!\s+constexpr)|else|switch|case)\b", b), blocks[-3:]
