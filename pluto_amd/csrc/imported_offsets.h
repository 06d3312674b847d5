// Where a lane of imported_several_kernel finds its sixteen bytes of a step, as the offsets
// of a buffer load.  Plain C++, so that the rule can be checked without a GPU.
#pragma once

#include <algorithm>
#include <cstdint>

namespace pluto_hip {

struct SeveralPlace {
  uint32_t lane;   // vector offset
  uint32_t step;   // scalar offset
};

// The step's 256 bytes of every row begin at `at`; the lane reads piece `block` of a row that
// begins at `row_start`.  What lies past the end of a row reads zero: the descriptor
// compares the vector offset with its size less the scalar one, which therefore stays within
// the one row that there is at least.
constexpr SeveralPlace several_place(uint32_t row_bytes, uint32_t row_start, uint32_t at, uint32_t block) {
  return {at + block * 16 < row_bytes ? row_start + block * 16 : 0x80000000u, std::min(at, row_bytes)};
}

}  // namespace pluto_hip
