"""Buffer stores of more than eight bytes at a scalar offset: such a store can still read its
data registers when the next instruction writes them, and the compiler keeps the two apart
only where the offset is no register.  No kernel source may contain one; the uniform part of
an address belongs in the vector offset.

Buffer accesses of any width at a scalar offset: a descriptor checks the lane's offset only, so
that such an access reaches past the descriptor's end wherever the lane's offset alone does
not say so.  None may be made through a descriptor that ends at the last row of a sequence;
those that there are stay within a record or a row whatever the lane holds."""
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


# Accesses whose scalar offset is a place in what the descriptor covers for every lane: file, its
# expression.  Rows that do not exist have a lane offset beyond the descriptor by themselves.
WITHIN = {
    ("gdn_backward_chunked.hip", "uniform"),         # Memory<false>: records of whole chunks
    ("dense_imported.hip", "place.step"),            # several_place: within the one row there is at least
    ("dense_imported.hip", "at + 64 * s"),           # a block of a row's columns, clamped to its last
    ("dense_imported.hip", "at + 64 * half"),
}
# Functions that pass a scalar offset on: which argument, and the descriptors it is used with.
PASSED_ON = {("gdn_scan.hip", "lds_dma_16"): (3, {"src.scratch"})}  # records of whole chunks


def scalar_offsets(text):
    """Scalar offsets other than 0 of all buffer accesses in `text`."""
    found = []
    for m in re.finditer(r"raw_(?:ptr_)?buffer_(load|store)_\w+\(", text):
        found.append(arguments(text, m.end() - 1)[3 if m.group(1) == "store" else 2])
    for m in re.finditer(r"buffer_(?:load|store)_(?:dword|ubyte|byte|short|ushort)\w*\s+([^\n\"\\]+)", text):
        found.append(m.group(1).split(",")[-1].split()[0])
    return [offset for offset in found if offset != "0"]


@pytest.mark.parametrize("path", SOURCES, ids=os.path.basename)
def test_buffer_accesses_at_a_scalar_offset_stay_within(path):
    name = os.path.basename(path)
    with open(path) as source:
        text = source.read()
    for (file, function), (argument, descriptors) in PASSED_ON.items():
        if name != file:
            continue
        for m in re.finditer(r"(?<!inline void )\b%s\(" % function, text):
            call = arguments(text, m.end() - 1)
            assert call[argument] == "0" or call[0] in descriptors, call
    passed = {"%3"} if any(file == name for file, _ in PASSED_ON) else set()
    assert [o for o in scalar_offsets(text) if (name, o) not in WITHIN and o not in passed] == []


def test_the_search_finds_every_width():
    assert scalar_offsets("x = __builtin_amdgcn_raw_buffer_load_b64(rows, at / 2,\n i * (8 * E), 0);") == ["i * (8 * E)"]
    assert scalar_offsets("__builtin_amdgcn_raw_buffer_store_b64(bits, rows, at, i * 8, 0);") == ["i * 8"]
    assert scalar_offsets('"buffer_load_dword v1, %[rsrc], s5 offen lds\\n\\t"') == ["s5"]
    assert scalar_offsets('"buffer_store_dwordx2 v[2:3], v1, s[0:3], s9 offen"') == ["s9"]
    assert not scalar_offsets('"buffer_load_dwordx4 v1, %[rsrc], 0 offen offset:16 lds"')
    assert not scalar_offsets("__builtin_amdgcn_raw_buffer_store_b64(bits, rows, at + i * 8, 0, 0);")
