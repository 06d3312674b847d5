"""Buffer stores of more than eight bytes at a scalar offset: such a store can still read its
data registers when the next instruction writes them, and the compiler keeps the two apart
only where the offset is no register.  No kernel source may contain one; the uniform part of
an address belongs in the vector offset."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pluto_amd", "csrc")
SOURCES = sorted(p for end in ("hip", "h", "inc") for p in glob.glob(os.path.join(CSRC, "*." + end)))


def arguments(text, start):
    """Top-level arguments of the call whose opening bracket is at `start`."""
    depth, current, found = 0, "", []
    for c in text[start:]:
        depth += (c in "([{") - (c in ")]}")
        if depth == 0:
            return found + [current.strip()]
        if c == "," and depth == 1:
            found.append(current.strip())
            current = ""
        elif not (c == "(" and depth == 1 and not current):
            current += c
    raise AssertionError("unbalanced brackets")


def scalar_offset_stores(text):
    calls = [arguments(text, m.end() - 1) for m in re.finditer(r"raw_(?:ptr_)?buffer_store_b(?:96|128)\(", text)]
    lines = re.findall(r"buffer_store_dwordx[34]\s+[^,]+,[^,]+,[^,]+,\s*([^\s,]+)", text)
    return [a for a in calls if a[3] != "0"] + [offset for offset in lines if offset != "0"]


@pytest.mark.parametrize("path", SOURCES, ids=os.path.basename)
def test_wide_buffer_stores_take_no_scalar_offset(path):
    with open(path) as source:
        assert scalar_offset_stores(source.read()) == []


def test_the_search_finds_both_forms():
    assert scalar_offset_stores("__builtin_amdgcn_raw_buffer_store_b128(f(a, b), rows,\n at, 128 * db, 0);")
    assert scalar_offset_stores('"buffer_store_dwordx4 v[0:3], v4, %[rsrc], s5 offen\\n\\t"')
    assert not scalar_offset_stores("__builtin_amdgcn_raw_buffer_store_b128(f(a, b), rows, at + 128 * db, 0, 0);")
