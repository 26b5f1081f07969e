// Which kernels a 2-D TM call runs on when no time block is set: workgroup
// tiles (tm2d_tile.h), or, where those measured slower, the in-place kernels of
// tm2d_highorder.hip (orders 4 to 8, Born).  Every family
// gives the same fields, receivers and snapshots bit for bit.  The figures are
// us per step of whole calls, tiles / other, fp32 unless noted; cells are
// padded cells of all shots.
#pragma once

#include "tm2d_device.h"

#include <cstdint>

namespace tide_hip {
namespace tm2d {

// Orders 4 to 8 in place.  Runs of few steps: a tile loop's set-up (a second
// state, packed profiles) takes 0.1 ms, an in-place step 12 us and more (order 4,
// 441 x 942 cells and 4 shots, 1 step with snapshots 168 / 99 us, 8 steps 30 / 44
// us per step; adjoint 2 steps 224 / 122, 5 steps 64 / 97).  fp64 forward of orders
// 6 and 8, whose halo of 5 and 7 cells a step leaves 22 x 54 and 18 x 50 cells of a
// tile: order 6 441 x 942 x 12 131 / 101, 1065 x 1065 x 4 102 / 96, but 700 x 700
// x 4 44 / 46; order 8 441 x 942 x 12 151 / 106, 700 x 700 x 4 54 / 48, but 360 x
// 380 x 4 21.9 / 22.7.
inline bool in_place_forward(int half, size_t elem, int64_t n_shots, int64_t numel, int64_t nt) {
  if (nt < 8) return true;
  const int64_t cells = n_shots * numel;
  return elem == 8 && ((half == 3 && cells >= 2500000) || (half == 4 && cells >= 600000));
}
inline bool in_place_adjoint(int64_t nt) { return nt < 4; }

// The Born forward in place, fp64 and many shots (whole Jacobian products of 192
// steps, ms): order 8 200 x 220 x 12 13.4 / 11.4, 600 x 620 x 8 43 / 36, but 1000 x
// 1000 x 2 23 / 25 and 150 x 150 x 8 6.4 / 8.4; order 6 100 x 100 x 64 16.2 / 14.6,
// but 300 x 320 x 8 10.5 / 13.4.
inline bool in_place_born(int half, size_t elem, int64_t n_shots, int64_t numel) {
  const int64_t cells = n_shots * numel;
  return elem == 8 && ((half == 4 && n_shots >= 8 && cells >= 600000) ||
                       (half == 3 && n_shots >= 16 && cells >= 1000000));
}

}  // namespace tm2d
}  // namespace tide_hip
