// Instantiation unit of the batch's MODWT tiles: element type float.
#include "batch_tile.h"

namespace wh {
template <>
int batch_tile_launch<float>(BatchPass pass, unsigned count, const BatchTileArgs& a,
                            hipStream_t st) {
  return batch_tile_launch_impl<float>(pass, count, a, st);
}
}  // namespace wh
