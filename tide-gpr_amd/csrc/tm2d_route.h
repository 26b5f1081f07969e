// Which kernels a 2-D TM call runs on when no time block is set: workgroup
// tiles (tm2d_tile.h), or, where those measured slower, wavefront tiles (order 2)
// or the in-place kernels of tm2d_highorder.hip (orders 4 to 8).  Every family
// gives the same fields, receivers and snapshots bit for bit.  The figures are
// us per step of whole calls, tiles / other, fp32 unless noted; cells are
// padded cells of all shots.
#pragma once

#include "tm2d_tile_launch.h"

#include <cstdint>

namespace tide_hip {
namespace tm2d {

// Order-2 forward on two-step wavefront tiles: calls that store both snapshot
// streams at full fp32 width in every step, between 4.5 million cells and what
// leaves their two state buffers (24 bytes a cell, 4 more for each per-shot
// coefficient) well inside the 256 MB last-level cache: 600 x 640 cells and 12
// shots 25.4 / 22.5; 768 x 800 and 12 39.4 / 35.3; 950 x 950 and 8 36.1 / 33.5; 441 x
// 942 and 12 26.2 / 24.8; 500 x 640 and 24 43 / 38.  Below and above tiles are as
// fast or faster (560 x 600 x 12 18.6 / 19.3; 640 x 800 x 16 34.5 / 38.9; 1065 x
// 1065 x 12 77 / 90), so are they with fewer than 6 shots (1300 x 1300 x 4 26.8 /
// 27.6), with small grids, whose border tiles weigh more (441 x 500 x 24 27.1 /
// 28.9), with BF16 or sampled snapshots, and where a run is so short that the
// wavefront path's many allocations weigh.
inline bool wavefront_forward(size_t elem, int64_t n_shots, int64_t numel, int64_t nt,
                              bool both_streams, int fmt, int64_t step_ratio,
                              int batched_coefficients) {
  const int64_t cells = n_shots * numel;
  return elem == 4 && both_streams && fmt == 1 && step_ratio == 1 && nt >= 64 && n_shots >= 6 &&
         numel >= 250000 && cells >= 4500000 &&
         cells * (24 + 4 * batched_coefficients) <= 185000000;
}

// Order-2 adjoint on three-step wavefront tiles: large fp32 calls whose shots
// fill workgroups of four, which share one FP64 gradient slice (tiles hold one
// per shot).  Per cell the tiles' time grows with the state, the wavefront tiles'
// falls with the share of border tiles; the line is cells x cells of a grid, with
// two gradients from full snapshots of every step: 1300 x 1300 cells and 4 shots
// (1.14e13) 41.3 / 38.9; 2081 x 2081 x 4 102 / 90; 1541 x 1541 x 8 115 / 109; 1065 x
// 1065 x 12 (1.5e13) 91 / 86; below it 1065 x 1065 x 8 (1.03e13) 57.7 / 59.1, 1065 x
// 1065 x 4 28.4 / 29.5, 800 x 800 x 16 66 / 70.  With fewer gradient bytes it lies
// higher: BF16 1541 x 1541 x 4 (2.3e13) 54.6 / 55.9, 2081 x 2081 x 4 (7.5e13) 94 /
// 91.  Groups of three shots and fewer gain at most 2 % (2100 x 2100 x 3 78.1 /
// 76.8); per-shot gradients have no shared slice (1000 x 1000 x 8 58 / 98).
inline bool wavefront_adjoint(size_t elem, int64_t n_shots, int64_t numel, int64_t nt,
                              int gradients, int fmt, int64_t step_ratio, bool per_shot) {
  const bool full = gradients == 2 && fmt == 1 && step_ratio == 1;
  const double weight = (double)n_shots * (double)numel * (double)numel;
  return elem == 4 && gradients > 0 && !per_shot && nt >= 64 &&
         balanced_group((int)n_shots, 4) == 4 && weight >= (full ? 1.1e13 : 5e13);
}

// Orders 4 to 8 in place.  Runs of few steps: a tile loop's set-up (a second
// state, packed profiles) takes 0.1 ms, an in-place step 12 us and more (order 4,
// 441 x 942 cells and 4 shots, 1 step with snapshots 168 / 99 us, 8 steps 30 / 44
// us per step; adjoint 2 steps 224 / 122, 5 steps 64 / 97).
// fp64 forward of orders 6 and 8, whose halo of 5 and 7 cells a step leaves 22 x 54
// and 18 x 50 cells of a tile.  Order 8 (one step per launch) takes about 6 us per
// round of workgroups, in place 19 us per million cells and 8 more than tiles at
// the start: 441 x 942 x 12 151 / 106, 700 x 700 x 4 54 / 48, 110 x 120 x 40 34 / 26,
// but 360 x 380 x 4 21.9 / 22.7, 64 x 200 x 40 27 / 28, 200 x 220 x 12 25.1 / 25.5.
// Order 6: large calls (441 x 942 x 12 131 / 101, 1065 x 1065 x 4 102 / 96, but 700 x
// 700 x 4 44 / 46), and many shots of grids with edge tiles only, 9 us a round (128
// x 128 x 64 45 / 33, 110 x 120 x 40 29 / 24, but 150 x 150 x 32 28 / 29, 64 x 200 x
// 40 21 / 26).
inline bool in_place_forward(int half, size_t elem, int64_t n_shots, int64_t numel, int64_t nt,
                             const TilePlan &plan, bool edge_tiles_only) {
  if (nt < 8) return true;
  if (elem == 4 || half < 3) return false;
  const double cells = 1e-6 * (double)n_shots * (double)numel;
  const int64_t rounds = ((int64_t)plan.n_xt * plan.n_yt * n_shots + 255) / 256;
  if (half == 4) return 6.0 * (double)rounds >= 8.5 + 19.0 * cells;
  return cells >= 2.5 || (plan.steps == 1 && edge_tiles_only &&
                          9.0 * (double)rounds >= 12.5 + 17.5 * cells + 0.1 * (double)n_shots);
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
