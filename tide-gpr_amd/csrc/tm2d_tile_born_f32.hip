// Launchers of the workgroup-tile Born kernels for float fields.
#define TIDE_TM2D_TILE_DEFINITIONS
#include "tm2d_tile_launch.h"

namespace tide_hip {
namespace tm2d {

template void launch_tile_born<float>(int, const TilePlan &, bool, hipStream_t,
                                      const TileBornArgs<float> &);

}  // namespace tm2d
}  // namespace tide_hip
