// Launch plan and launchers of the workgroup-tile kernels (tm2d_tile.h).
// The definitions compile in one translation unit per pass and field type
// (tm2d_tile_{fwd,adj,born}_{f32,f64}.hip).
#pragma once

#include "tm2d_tile.h"

#include <algorithm>
#include <cmath>

namespace tide_hip {
namespace tm2d {

struct TilePlan {
  int waves, rows, steps;  // wavefronts per workgroup, rows per wavefront, steps per launch
  int halo, own_rows, own_cols, n_xt, n_yt;
};

inline TilePlan make_tile_plan(int half, int ny, int nx, int waves, int rows, int steps) {
  TilePlan p;
  p.waves = waves;
  p.rows = rows;
  p.steps = steps;
  p.halo = steps * (2 * half - 1);
  p.own_rows = waves * rows - 2 * p.halo;
  p.own_cols = 64 - 2 * p.halo;
  p.n_xt = (nx + p.own_cols - 1) / p.own_cols;
  p.n_yt = (ny + p.own_rows - 1) / p.own_rows;
  return p;
}

// The tiles of a plan that meet no grid edge and no CPML strip (see
// tile_place); half is the stencil half-width.
template <typename T> TileOrder tile_order(const TilePlan &p, const Geom<T> &g, int half) {
  auto inner = [&](int n_tiles, int own, int len, int n, int pml0, int pml1h, int &a, int &b) {
    a = b = 0;
    for (int t = 0; t < n_tiles; ++t) {
      const int c0 = t * own - p.halo, c1 = c0 + len - 1;
      if (c0 < half || c1 > n - half - 1 || c0 < pml0 || c1 >= pml1h) continue;
      if (a == b) a = t;
      b = t + 1;
    }
  };
  TileOrder o;
  o.n_yt = p.n_yt;
  inner(p.n_xt, p.own_cols, 64, g.nx, g.pml_x0, g.pml_x1h, o.xa, o.xb);
  inner(p.n_yt, p.own_rows, p.waves * p.rows, g.ny, g.pml_y0, g.pml_y1h, o.ya, o.yb);
  if (o.xa == o.xb || o.ya == o.yb) o.xa = o.xb = o.ya = o.yb = 0;
  return o;
}

// Duration of one launch of `steps` steps when every workgroup runs at once
// (one per CU), in microseconds: start, loads and stores plus the steps.
// Measured on 60^2 to 150 x 200 grids; half is the stencil half-width.
template <typename T>
double tile_launch_us(int half, int rows, int steps, bool adjoint, bool storing) {
  if (sizeof(T) == 8)
    return adjoint ? (rows == 2 ? 11.2 + 1.8 * steps : 22.0 + 6.0 * steps)
                   : (rows == 2 ? 9.8 + 1.5 * steps : 12.0 + 3.0 * steps);
  if (adjoint) {
    if (rows == 2) return 9.2 + 1.7 * steps;
    return (half == 1 ? 13.0 : 17.0) + (half <= 2 ? 3.0 : 5.0) * steps;
  }
  if (rows == 2) return 6.4 + (storing ? 1.2 : 0.9) * steps;
  return storing ? 6.8 + 2.0 * steps : 9.1 + 1.3 * steps;
}

// Tile shape and steps per launch of a problem: the shape with the least time
// per step, a launch taking as many rounds of workgroups as its tiles fill the
// CUs.  Small problems want small tiles (many CUs at work, few rows per
// wavefront) and many steps (a launch's start is paid once); once the tiles
// outnumber the CUs, larger tiles with less halo.  Measured against the model
// (fp32, order 2, us per step, forward / adjoint): 171 000 cells 2.1 / 3.5
// with 32-row tiles of 8 steps (64-row: 2.8 / 5.1), 577 000 cells 3.3 / 5.7
// with 64-row tiles of 6 (32-row: 4.5 / 7.6).
template <typename T>
TilePlan plan_tiles(int half, int ny, int nx, int n_shots, bool adjoint, bool storing) {
  constexpr int kCus = 256;
  TilePlan best{};
  double best_us = 1e30;
  for (int rows = 2; rows <= 4; rows += 2) {
    // a wavefront holds at least `half` rows (it exchanges that many), and
    // 64-row tiles of doubles overflow the registers of 16 wavefronts
    if (rows < half || (sizeof(T) == 8 && rows == 4 && half <= 2)) continue;
    const int waves = rows == 4 && (sizeof(T) == 8 || (adjoint && half == 4)) ? 8 : kTileWaves;
    for (int steps = 1; steps <= kTileSteps; ++steps) {
      const int halo = steps * (2 * half - 1);
      // at least a quarter of the tile's rows and half its columns owned
      if (halo > 16 || waves * rows - 2 * halo < waves * rows / 4) break;
      const TilePlan p = make_tile_plan(half, ny, nx, waves, rows, steps);
      const double n = (double)p.n_xt * p.n_yt * n_shots;
      const double rounds = n <= kCus ? 1.0 : std::min(std::ceil(n / kCus), n / kCus + 0.3);
      const double us = rounds * tile_launch_us<T>(half, rows, steps, adjoint, storing) / steps;
      if (us < best_us) {
        best_us = us;
        best = p;
      }
    }
  }
  return best;
}

// The Born kernel's tiles: 32 rows (two field sets fill the registers that one
// takes in a 64-row tile), by 16 wavefronts of 2 rows in fp32 up to order 4, else
// by 8 of 4 (wide stencils exchange up to 4 rows; two sets of doubles need the
// 256 registers of 8 wavefronts, and their LDS rows fit 160 KB).
constexpr int kBornRows = 32;
template <typename T> constexpr int born_rows(int half) {
  return sizeof(T) == 4 && half <= 2 ? 2 : 4;
}

template <typename T> TilePlan plan_born(int half, int ny, int nx, int n_shots) {
  const int rows = born_rows<T>(half), waves = kBornRows / rows;
  TilePlan best{};
  double best_us = 1e30;
  for (int steps = 1; steps <= kTileSteps; ++steps) {
    const int halo = steps * (2 * half - 1);
    if (kBornRows - 2 * halo < kBornRows / 4) break;
    const TilePlan p = make_tile_plan(half, ny, nx, waves, rows, steps);
    const double rounds = std::max(1.0, (double)p.n_xt * p.n_yt * n_shots / 256.0);
    const double us = std::min(std::ceil(rounds), rounds + 0.3) *
                      (10.0 + (rows == 2 ? 1.8 : 3.0) * steps) / steps;
    if (us < best_us) {
      best_us = us;
      best = p;
    }
  }
  return best;
}

// Steps of each launch of a time loop of nt steps, at most `most` each: the
// fewest launches, an even number of them where nt allows it (the state ping-
// pongs between the caller's arrays and a scratch copy, and an even count ends
// in the caller's arrays), as equal as possible.
struct LaunchSteps {
  int64_t nt, launches;
  LaunchSteps(int64_t nt_, int most) : nt(nt_), launches((nt_ + most - 1) / most) {
    if ((launches & 1) && nt > launches) ++launches;
  }
  int at(int64_t k) const { return (int)(nt * (k + 1) / launches - nt * k / launches); }
  bool ends_in_scratch() const { return (launches & 1) != 0; }
};

// Of the calling thread: whether a call whose tile loop has no room goes on
// with the kernels that need less scratch (else it returns kOutOfMemory, and a
// caller that holds device memory unused may release it and call again), and
// the most scratch of a tile loop in bytes.
extern thread_local bool tile_fallback;
extern thread_local size_t tile_scratch_limit;

template <typename T>
void launch_tile_fwd(int half, const TilePlan &p, int fmt, hipStream_t stream, const TileFwdArgs<T> &a);
template <typename T>
void launch_tile_adj(int half, const TilePlan &p, int fmt, hipStream_t stream, const TileAdjArgs<T> &a);
template <typename T>
void launch_tile_born(int half, const TilePlan &p, bool store, hipStream_t stream, const TileBornArgs<T> &a);

// Several order-2 fp32 problems of tile shape p: `grid` workgroups.
void launch_tile_fwd_items(const TilePlan &p, int fmt, int64_t grid, hipStream_t stream,
                           const TileFwdArgs<float> *table, const int32_t *tile_item);
void launch_tile_adj_items(const TilePlan &p, int fmt, int64_t grid, hipStream_t stream,
                           const TileAdjArgs<float> *table, const int32_t *tile_item);

#ifdef TIDE_TM2D_TILE_DEFINITIONS

template <typename T, int P, int R, int W>
void tile_fwd_fmt(const TilePlan &p, int fmt, hipStream_t stream, const TileFwdArgs<T> &a) {
  const dim3 block(64, (unsigned)p.waves);
  const unsigned grid = (unsigned)((int64_t)p.n_xt * p.n_yt * a.n_shots);
  const size_t lds = TileRows<T, P>::bytes(p.waves, a.steps);
  if (fmt == 0) return tile_fwd<T, P, R, W, 0><<<grid, block, lds, stream>>>(a);
  if constexpr (sizeof(T) == 4)
    if (fmt == 2) return tile_fwd<T, P, R, W, 2><<<grid, block, lds, stream>>>(a);
  tile_fwd<T, P, R, W, 1><<<grid, block, lds, stream>>>(a);
}

template <typename T, int P, int R, int W>
void tile_adj_fmt(const TilePlan &p, int fmt, hipStream_t stream, const TileAdjArgs<T> &a) {
  const dim3 block(64, (unsigned)p.waves);
  const unsigned grid = (unsigned)((int64_t)p.n_xt * p.n_yt * a.n_shots);
  const size_t lds = TileRows<T, P>::bytes(p.waves, a.steps);
  if (fmt == 0) return tile_adj<T, P, R, W, 0><<<grid, block, lds, stream>>>(a);
  if constexpr (sizeof(T) == 4)
    if (fmt == 2) return tile_adj<T, P, R, W, 2><<<grid, block, lds, stream>>>(a);
  tile_adj<T, P, R, W, 1><<<grid, block, lds, stream>>>(a);
}

// The shapes plan_tiles() picks from.
#define TIDE_TILE_PICK(fn)                                             \
  if constexpr (P <= 2) {                                              \
    if (p.rows == 2) return fn<T, P, 2, kTileWaves>(p, fmt, stream, a); \
  }                                                                    \
  if constexpr (sizeof(T) == 4) {                                      \
    if (p.waves > 8) return fn<T, P, 4, kTileWaves>(p, fmt, stream, a); \
  }                                                                    \
  if constexpr (P > 2) return fn<T, P, 4, 8>(p, fmt, stream, a);

template <typename T, int P>
void tile_fwd_shape(const TilePlan &p, int fmt, hipStream_t stream, const TileFwdArgs<T> &a) {
  TIDE_TILE_PICK(tile_fwd_fmt)
}
template <typename T, int P>
void tile_adj_shape(const TilePlan &p, int fmt, hipStream_t stream, const TileAdjArgs<T> &a) {
  TIDE_TILE_PICK(tile_adj_fmt)
}

template <typename T>
void launch_tile_fwd(int half, const TilePlan &p, int fmt, hipStream_t stream, const TileFwdArgs<T> &a) {
  switch (half) {
    case 1: tile_fwd_shape<T, 1>(p, fmt, stream, a); break;
    case 2: tile_fwd_shape<T, 2>(p, fmt, stream, a); break;
    case 3: tile_fwd_shape<T, 3>(p, fmt, stream, a); break;
    default: tile_fwd_shape<T, 4>(p, fmt, stream, a); break;
  }
}
template <typename T>
void launch_tile_adj(int half, const TilePlan &p, int fmt, hipStream_t stream, const TileAdjArgs<T> &a) {
  switch (half) {
    case 1: tile_adj_shape<T, 1>(p, fmt, stream, a); break;
    case 2: tile_adj_shape<T, 2>(p, fmt, stream, a); break;
    case 3: tile_adj_shape<T, 3>(p, fmt, stream, a); break;
    default: tile_adj_shape<T, 4>(p, fmt, stream, a); break;
  }
}

template <typename T, int P>
void tile_born_shape(const TilePlan &p, bool store, hipStream_t stream, const TileBornArgs<T> &a) {
  constexpr int R = born_rows<T>(P), W = kBornRows / R;
  const dim3 block(64, (unsigned)p.waves);
  const unsigned grid = (unsigned)((int64_t)p.n_xt * p.n_yt * a.n_shots);
  const size_t lds = 2 * TileRows<T, P>::bytes(p.waves, a.steps);
  if (store)
    tile_born<T, P, R, W, true><<<grid, block, lds, stream>>>(a);
  else
    tile_born<T, P, R, W, false><<<grid, block, lds, stream>>>(a);
}

template <typename T>
void launch_tile_born(int half, const TilePlan &p, bool store, hipStream_t stream, const TileBornArgs<T> &a) {
  switch (half) {
    case 1: tile_born_shape<T, 1>(p, store, stream, a); break;
    case 2: tile_born_shape<T, 2>(p, store, stream, a); break;
    case 3: tile_born_shape<T, 3>(p, store, stream, a); break;
    default: tile_born_shape<T, 4>(p, store, stream, a); break;
  }
}

#endif  // TIDE_TM2D_TILE_DEFINITIONS

}  // namespace tm2d
}  // namespace tide_hip
