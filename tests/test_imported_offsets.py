"""The offsets of the imported projections' buffer loads for two to eight tokens, compiled for
the host: a scalar offset never exceeds the descriptor's size (the hardware compares the
vector offset with the difference), a piece that exists is read where it lies, and any
other lies past the end, which reads zero."""
import shutil
import subprocess

import pytest

from pluto_amd import build

PROGRAM = r"""
#include "imported_offsets.h"
#include <cstdio>
int main() {
  using pluto_hip::several_place;
  for (unsigned row_bytes = 128; row_bytes <= 2 * 9216; row_bytes += 128)
    for (unsigned rows = 1; rows <= 4; ++rows) {
      const unsigned long long size = 1ull * rows * row_bytes;
      for (unsigned step = 0; step < 96; ++step)       // of four panels of 24
        for (unsigned lane = 0; lane < 64; ++lane) {
          const unsigned row = lane % 4, block = lane / 4, at = step * 256;
          const auto place = several_place(row_bytes, row * row_bytes, at, block);
          if (place.step > size) return std::printf("scalar %u %u %u\n", row_bytes, rows, step), 1;
          const bool exists = row < rows && at + block * 16 < row_bytes;
          const bool read = place.lane + 16ull <= size - place.step;
          if (exists != read) return std::printf("range %u %u %u %u\n", row_bytes, rows, step, lane), 1;
          if (exists && 1ull * place.lane + place.step != 1ull * row * row_bytes + at + block * 16)
            return std::printf("place %u %u %u %u\n", row_bytes, rows, step, lane), 1;
        }
    }
  std::puts("ok");
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_offsets_stay_within_the_descriptor(tmp_path):
    source, program = tmp_path / "offsets.cc", tmp_path / "offsets"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++20", "-I" + build.CSRC, str(source), "-o", str(program)], check=True)
    done = subprocess.run([str(program)], stdout=subprocess.PIPE, text=True)
    assert done.returncode == 0, done.stdout
    assert done.stdout == "ok\n"
