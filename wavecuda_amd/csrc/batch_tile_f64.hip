// Instantiation unit of the batch's MODWT tiles: element type double.
#include "batch_tile.h"

namespace wh {
template <>
int batch_tile_launch<double>(BatchPass pass, unsigned count, const BatchTileArgs& a,
                            hipStream_t st) {
  return batch_tile_launch_impl<double>(pass, count, a, st);
}
}  // namespace wh
