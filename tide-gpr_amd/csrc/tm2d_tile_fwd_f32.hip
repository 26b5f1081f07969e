// Launchers of the workgroup-tile fwd kernels for float fields.
#define TIDE_TM2D_TILE_DEFINITIONS
#include "tm2d_tile_launch.h"

namespace tide_hip {
namespace tm2d {

template void launch_tile_fwd<float>(int, const TilePlan &, int, hipStream_t,
                                   const TileFwdArgs<float> &);

template <int R>
static void items_shape(const TilePlan &p, int fmt, int64_t grid, hipStream_t stream,
                        const TileFwdArgs<float> *table, const int32_t *tile_item) {
  const dim3 block(64, (unsigned)p.waves);
  const size_t lds = TileRows<float, 1>::bytes(p.waves, p.steps);
  if (fmt == 0)
    tile_fwd_items<float, 1, R, kTileWaves, 0><<<(unsigned)grid, block, lds, stream>>>(table, tile_item);
  else if (fmt == 2)
    tile_fwd_items<float, 1, R, kTileWaves, 2><<<(unsigned)grid, block, lds, stream>>>(table, tile_item);
  else
    tile_fwd_items<float, 1, R, kTileWaves, 1><<<(unsigned)grid, block, lds, stream>>>(table, tile_item);
}

void launch_tile_fwd_items(const TilePlan &p, int fmt, int64_t grid, hipStream_t stream,
                           const TileFwdArgs<float> *table, const int32_t *tile_item) {
  if (p.rows == 2) items_shape<2>(p, fmt, grid, stream, table, tile_item);
  else items_shape<4>(p, fmt, grid, stream, table, tile_item);
}

}  // namespace tm2d
}  // namespace tide_hip
