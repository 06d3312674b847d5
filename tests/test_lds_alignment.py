"""Arrays of single numbers in LDS that are read or written several at a time: the compiler
places an array of floats at any multiple of four bytes, a 16-byte access needs one of 16.
Such an array's declaration says so."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pluto_amd", "csrc")
SOURCES = sorted(p for end in ("hip", "h") for p in glob.glob(os.path.join(CSRC, "*." + end)))
NUMBERS = r"(?:float|int|uint32_t|uint16_t|unsigned char)"


def wide_accesses(text):
    """Names of such arrays that are accessed wide in the function that declares them."""
    found = []
    for declaration in re.finditer(r"__shared__ (%s [^;]*);" % NUMBERS, text):
        function = text[declaration.end():].split("\n}\n")[0]
        for name in re.findall(r"(\w+)\[", re.sub(r"\[[^\]]*\]", "[", declaration.group(1))):
            if re.search(r"reinterpret_cast<[^>]*(?:2|4|x4|x8)\s*\*>\(\s*&?%s\b" % name, function):
                found.append(name)
    return found


@pytest.mark.parametrize("path", SOURCES, ids=os.path.basename)
def test_wide_accesses_have_aligned_arrays(path):
    with open(path) as source:
        assert wide_accesses(source.read()) == []


def test_the_search_finds_them():
    use = "float4 v = *reinterpret_cast<const float4*>(&rows[p][0][16 * r]);\n}\n"
    assert wide_accesses("__shared__ float rows[2][2][128];\n" + use) == ["rows"]
    assert wide_accesses("__shared__ float parts[2], rows[4];\n" + use) == ["rows"]
    assert not wide_accesses("__shared__ __attribute__((aligned(16))) float rows[2][2][128];\n" + use)
    assert not wide_accesses("__shared__ float rows[2];\n}\n" + use)
