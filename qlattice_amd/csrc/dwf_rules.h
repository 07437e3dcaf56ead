// Rules of the host code that depend on sizes alone: plain C++, so that they
// can be tested without a GPU.
#pragma once

#include <cstddef>
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
// cost 1 to 2%, there and below the FP32 hop by itself 3 to 9%; the FP64 hop by
// itself is faster with 8 planes at 24^3x64 Ls12 (0.73 against 0.78 ms).
inline int z_tile(int xh, int by, int nz)
{
  auto whole_lines = [&](int b) { return (int64_t)xh * by * b % 8 == 0; };
  auto far = [](int b) { return b * b > 97 ? b * b / 97.0 : 97.0 / (b * b); };
  int best = nz;
  for (int b = nz - 1; b > 0; --b)
    if (nz % b == 0 && (whole_lines(b) || !whole_lines(nz)) && far(b) < far(best)) best = b;
  return best;
}

// Sites per block of the three-phase kernels where the autotuner does not
// choose them (single columns, fixed tiles), half volume vh.  16 makes whole
// waves of four rows, with the s-matrix phase on the matrix cores; Ls that is
// no multiple of 4 needs 32.  Mpc^+ Mpc of one column, us:
//   Ls 12, 16 against 32 sites: FP32 42 / 46 at 8^3x16, 262 / 267 at 16^3x32,
//     FP16 storage 37 / 41 and 166 / 179; 20^3x40 FP32 742 / 706
//   Ls 16: FP32 48 / 55 and 326 / 326, FP16 storage 42 / 48 and 201 / 210
//   Ls 8, where a block of 16 sites is only two waves: FP32 38.1 / 38.6 at
//     8^3x16, 86 / 79 at 12^3x24, 188 / 174 at 16^3x32, FP16 storage 34.3 /
//     34.6, 65 / 60 and 123 / 115, with four columns 51 / 50, 152 / 144, 388 /
//     369; 16 is ahead only in FP32 at some 300 blocks of 32 (12^4: 55 / 58)
//   Ls 24, 16 against 8 sites (six waves and 41 KB of LDS against three and
//     23 KB, so three blocks a CU against six): FP32 57 / 63 at 8^3x16, 89 /
//     96 at 8^3x32, 124 / 124 at 12^4, 172 / 153 at 12^3x16, 577 / 525 at
//     16^3x32, FP16 storage 49 / 53, 69 / 72, 96 / 91, 136 / 109 and 422 /
//     360: 8 from more than two blocks of 16 sites a CU on
inline int three_phase_sites(int ls, int64_t vh)
{
  if (ls == 8) return 32;
  if (ls == 24) return vh > 2 * 256 * 16 ? 8 : 16;
  return ls % 4 ? 32 : 16;
}

// Whether the staging ring of the host copies is to be made for a transfer of
// `bytes` after `without` transfers that went without one.  Its 16 MB of
// pinned memory cost up to 2 ms, more than one call on a small array wins
// back: M_ee on host half fields on a new inverter, first call with a ring
// against the runtime's copies 2.9 against 1.2 ms at 12.6 MB, 3.6 against 2.4
// ms at 25 MB, 5.4 against 3.1 ms at 32 MB, 3.1 to 5.5 against 4.7 to 6.6 ms at
// 48 MB; the calls after it 0.90 / 1.11, 1.50 / 2.2, 2.1 / 2.9 and 2.7 to 5.8 /
// 4.6 to 6.5 ms.  So a first call, one array in and one out, goes without, and
// the next one is taken for the second of many.
inline bool ring_pays(size_t bytes, int without) { return bytes >= (size_t)40 << 20 || without >= 2; }

}  // namespace qdwf
