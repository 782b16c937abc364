// Instantiation unit of the MODWT tile kernels: element type float.
#include "modwt_tile.h"

namespace wh {
template <>
int modwt_tile_launch<float>(TileOp op, int filt, const GroupLaunch& gl, const ModwtArgs& a,
                              const GradArgs& q, hipStream_t st) {
  return modwt_tile_launch_impl<float>(op, filt, gl, a, q, st);
}
}  // namespace wh
