// Launchers of the workgroup-tile fwd kernels for float fields.
#define TIDE_TM2D_TILE_DEFINITIONS
#include "tm2d_tile_launch.h"

namespace tide_hip {
namespace tm2d {

template void launch_tile_fwd<float>(int, const TilePlan &, int, hipStream_t,
                                   const TileFwdArgs<float> &);

}  // namespace tm2d
}  // namespace tide_hip
