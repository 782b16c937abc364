// Instantiation unit of the MODWT tile kernels: element type double.
#include "modwt_tile.h"

namespace wh {
template <>
int modwt_tile_launch<double>(bool inverse, int filt, const GroupLaunch& gl, const ModwtArgs& a,
                             hipStream_t st) {
  return modwt_tile_launch_impl<double>(inverse, filt, gl, a, st);
}
}  // namespace wh
