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

// Planes of a z tile of the device site order (dwf_common.h): the divisor of
// Z closest in ratio to 10, so that a t step of a tile is short enough for
// the L2 to keep the neighbouring time slices.  A t neighbour is X/2*by*bz
// sites away; where the whole Z makes that a multiple of 8 (a 128-byte line
// holds 8 sites of a slot) only tiles that do so too are taken: with others
// every t gather of a wave touches one line more.  Measured against no tiles,
// Mpc^+ Mpc at Ls 12, FP64 / FP32 one column / FP16 storage four columns:
//   24^3x64, 12 planes 0.94 / 0.93 / 1.00, 8 planes 0.94 / 0.96 / 1.03
//   32^4, 8 planes 0.90 / 0.92 / 1.01, 16 planes 0.97 / 0.96 / 1.02
//   28^3x32, 4 planes 0.93 / 0.95 / 1.00, 7 (686 sites) 0.99 / 0.98 / 1.02
//   20^3x40, 4 planes 0.97 / 1.01 / 1.06, 10 (500 sites) 1.00 / 1.02 / 1.02
//   16^3x32, 8 planes 0.95 / 0.99 / 0.96
//   14^3x28, 7 planes 0.97 / 1.00 / 0.98
// (the square of the middle is 97: 12 planes before 8, 7 before 14, none
// before 4 at Z = 20).  On lattices that fit the L2s anyway (6x10x14x22) tiles
// cost 1 to 2%, and the FP32 hop by itself 1 to 5%.
inline int z_tile(int xh, int by, int nz)
{
  auto whole_lines = [&](int b) { return (int64_t)xh * by * b % 8 == 0; };
  auto far = [](int b) { return b * b > 97 ? b * b / 97.0 : 97.0 / (b * b); };
  int best = nz;
  for (int b = nz - 1; b > 0; --b)
    if (nz % b == 0 && (whole_lines(b) || !whole_lines(nz)) && far(b) < far(best)) best = b;
  return best;
}

}  // namespace qdwf
