// Grid of the GEMM tile kernels.  HIP launches no grid dimension of 2^32
// work-items or more, which the tiles of a tall product pass (64 x 64 tiles of
// 512 threads: 2^29 rows), so tiles beyond 2^22 go to the grid's third
// dimension: workgroup (x, z) takes tile z * 2^22 + x, and those past the last
// tile leave at once.
#pragma once

#include "layout_maps.h"

namespace ipus {

constexpr uint32_t kTileGridX = 1u << 22;  // a multiple of the 8 XCDs; 2^31 work-items of 512 threads

struct TileGrid {
  uint32_t x, z;
};

// tiles: at least 1 and below 2^31.
inline TileGrid tile_grid(uint64_t tiles) {
  if (tiles <= kTileGridX) return {(uint32_t)tiles, 1};
  return {kTileGridX, (uint32_t)((tiles + kTileGridX - 1) / kTileGridX)};
}

IPUS_HD uint32_t grid_tile(uint32_t x, uint32_t z) { return z * kTileGridX + x; }

}  // namespace ipus
