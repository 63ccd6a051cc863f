// The tiled batched GEMV's kernels for W4 (wq_tile.h).
#include "wq_tile.h"

namespace agq {

int tile_launch_w4(const TileArgs& a, const TileShape& t, const void* x, int k, int group, int act, uint8_t* img,
                   hipStream_t s) {
  return group == 128 ? tile_launch<4, 128>(a, t, x, k, act, img, s) : tile_launch<4, 64>(a, t, x, k, act, img, s);
}

}  // namespace agq
