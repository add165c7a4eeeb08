"""Rules of the kernel sources that no result shows, read from the sources on the CPU."""
import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "castforge_amd" / "csrc"


def _args(text: str, start: int) -> list[str]:
    """The arguments of the call whose '(' is at start."""
    depth, out, cur = 0, [], ""
    for c in text[start:]:
        if c in "([{":
            depth += 1
        elif c in ")]}":
            depth -= 1
        if depth == 0:
            return out + [cur.strip()]
        if c == "," and depth == 1:
            out.append(cur.strip())
            cur = ""
        elif depth > 1 or c != "(":
            cur += c
    raise AssertionError("unbalanced call")


@pytest.mark.parametrize("src", sorted(p.name for p in CSRC.glob("*.hip")))
def test_rows_are_in_the_range_checked_offset(src):
    """A buffer load's scalar offset takes no part in the range check (or makes it wrap): the row of an
    operand, a multiple of K, is in the vector offset, so that rows past M and N are not read."""
    text = (CSRC / src).read_text()
    for m in re.finditer(r"__builtin_amdgcn_raw_(ptr_)?buffer_load_(lds|b\d+)\(", text):
        args = _args(text, m.end() - 1)
        scalar = args[4] if m.group(2) == "lds" else args[2]
        line = text.count("\n", 0, m.start()) + 1
        assert not re.search(r"\b(K|row\w*)\b", scalar), f"{src}:{line}: row in the scalar offset: {scalar}"
