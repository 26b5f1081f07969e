// Launchers of the workgroup-tile Born kernels for double fields.
#define TIDE_TM2D_TILE_DEFINITIONS
#include "tm2d_tile_launch.h"

namespace tide_hip {
namespace tm2d {

template void launch_tile_born<double>(int, const TilePlan &, bool, hipStream_t,
                                      const TileBornArgs<double> &);

}  // namespace tm2d
}  // namespace tide_hip
