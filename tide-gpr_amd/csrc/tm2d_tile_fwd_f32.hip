// Launchers of the workgroup-tile fwd kernels for float fields.
#define TIDE_TM2D_TILE_DEFINITIONS
#include "tm2d_tile_launch.h"

namespace tide_hip {
namespace tm2d {

template void launch_tile_fwd<float>(int, const TilePlan &, int, hipStream_t,
                                   const TileFwdArgs<float> &);

void launch_tile_fwd_items(const TilePlan &p, int fmt, int64_t grid, hipStream_t stream,
                           const TileFwdArgs<float> *table, const int32_t *tile_item) {
  using Kernel = void (*)(const TileFwdArgs<float> *, const int32_t *);
  static const Kernel kernels[2][3] = {  // by rows per wavefront (2, 4) and snapshot format
      {tile_fwd_items<float, 1, 2, kTileWaves, 0>, tile_fwd_items<float, 1, 2, kTileWaves, 1>,
       tile_fwd_items<float, 1, 2, kTileWaves, 2>},
      {tile_fwd_items<float, 1, 4, kTileWaves, 0>, tile_fwd_items<float, 1, 4, kTileWaves, 1>,
       tile_fwd_items<float, 1, 4, kTileWaves, 2>}};
  kernels[p.rows == 2 ? 0 : 1][fmt]<<<(unsigned)grid, dim3(64, (unsigned)p.waves),
                                      TileRows<float, 1>::bytes(p.waves, p.steps), stream>>>(
      table, tile_item);
}

}  // namespace tm2d
}  // namespace tide_hip
