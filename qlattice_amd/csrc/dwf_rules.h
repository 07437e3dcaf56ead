// Rules of the host code that depend on sizes alone: plain C++, so that they
// can be tested without a GPU.
#pragma once

#include <cstdint>

namespace qdwf {

// Blocks of a launch with one thread per element.  A grid dimension takes
// fewer than 2^32 threads (the QED operator has that many from 64 GiB per
// field on: 128^3x64 Ls8), so a launch beyond it is spread over y.  Block (x,
// y) is number y * g.x + x; fewer than y of the last ones have no elements.
struct Grid2 {
  unsigned x, y;
};
inline Grid2 split_blocks(int64_t nblk, int block)
{
  const int64_t most = (((int64_t)1 << 32) - 1) / block;
  const int64_t y = (nblk + most - 1) / most;
  return Grid2{(unsigned)((nblk + y - 1) / y), (unsigned)y};
}

}  // namespace qdwf
