// Instantiation unit of the MODWT tile kernels: element type float.
#include "modwt_tile.h"

namespace wh {
template <>
int modwt_tile_launch<float>(bool inverse, int filt, const GroupLaunch& gl, const ModwtArgs& a,
                             hipStream_t st) {
  return modwt_tile_launch_impl<float>(inverse, filt, gl, a, st);
}
}  // namespace wh
