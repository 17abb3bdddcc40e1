// Which kernel runs a GEMM: models of their times.  Plain C++, so that a host
// program can check the choice.
#pragma once

#include <stdint.h>

#include <cmath>

namespace ipus {

// What every row pitch and address of fp16 operands allows; kElement (also K = 0 and
// operands past the DMA's buffer ranges) has no 256 x 256 tile.
enum class GemmAccess { kChunk, kDword, kElement };  // 16, 4, 2 bytes

// Modelled time of each tile size, us, fitted to launches timed on the chip: a
// start-up, and per round of 256 tiles a fixed part (first operand tiles, store
// of C) and one per 64-k step (32 x 32 tiles: 128-k).  A 256 x 256 round costs
// more the more of its CUs work (C to memory, the power limit).  Kernel times
// (256 x 256, 128 x 128, 64 x 64, 32 x 32) of M x N x K:
//   4096 x 4096 x 64     11.1  17.8  22.8  60.8    2048 x 2048 x 64   7.9  5.9  7.5 16.8
//   4096 x 4096 x 1024   30.4  39.1  55.8   130    2048 x 2048 x 1024 22.5 10.6 14.8 34.2
//   2592 x 4368 x 440    18.6  22.8  29.3  66.2    1024 x 1024 x 64   7.3  5.1  3.4  5.7
//   3072 x 3072 x 128     9.3  14.6  15.4  34.6    1024 x 1024 x 2048 35.5 15.4  7.8 15.9
//   3093 x 1976 x 640    17.6  16.3  19.2  40.9    256 x 256 x 1024   21.2  8.6  5.2  4.0
// (a model without the fixed part of a round had taken small tiles for many
// short sums: 4096 x 4096 x 64 22.8, 2592 x 4368 x 440 27.2).  kElements, whose loads
// pass through registers: 4095 x 4097 x 441 45.5 (128 x 128) 56.1 136, 1023 x 1025 x
// 65 6.4 4.9 7.9, and past the buffer ranges 32 x 49152 x 49152 1,027 on 64 x 64, 1,290
// on 32 x 32.  The choice does not depend on the epilogue, so a fused epilogue gives
// the bits of the separate kernels.
inline uint32_t gemm_f16_tile(uint32_t rows, uint32_t columns, uint32_t inner, uint64_t batches, GemmAccess access) {
  struct Class {
    uint32_t tile;
    double start_us, round_us, step_us, element_step_us;
  };
  constexpr Class kClasses[] = {{128, 1.7, 3.6, 0.40, 0.90}, {64, 2.2, 1.2, 0.152, 0.33}, {32, 2.0, 0.75, 0.155, 0.55}};
  auto tiles_of = [&](uint32_t tile) {
    return (double)(((uint64_t)rows + tile - 1) / tile) * (double)(((uint64_t)columns + tile - 1) / tile) * (double)batches;
  };
  uint32_t best = 0;
  double best_us = 0;
  if (access != GemmAccess::kElement) {
    const double steps = (double)(((uint64_t)inner + 63) / 64), rounds = tiles_of(256) / 256, whole = std::floor(rounds);
    auto round_us = [&](double part) { return 6.0 + 2.9 * part + steps * (0.88 + 0.45 * part * part * part); };
    best = 256;
    best_us = whole * round_us(1.0) + (rounds > whole ? round_us(rounds - whole) : 0.0);
    if (access == GemmAccess::kDword) best_us += 3.5 * std::ceil(rounds);  // C stored by element
  }
  for (const Class& c : kClasses) {
    const uint32_t step = c.tile == 32 ? 128 : 64;
    const double steps = (double)(((uint64_t)inner + step - 1) / step), tiles = tiles_of(c.tile);
    // Two workgroups of the smaller tiles share a CU.
    const double rounds = tiles <= 256 ? 1.0 : c.tile >= 128 ? std::ceil(tiles / 256) : 2.0 * std::ceil(tiles / 512);
    const double us = c.start_us + rounds * (c.round_us + steps * (access == GemmAccess::kElement ? c.element_step_us : c.step_us));
    if (best == 0 || us < best_us) {
      best = c.tile;
      best_us = us;
    }
  }
  return best;
}

// Modelled time of the kernels, us, as gemm_f16_tile's: a start-up, and per round
// of 256 tiles a fixed part and one per 32-k step (32 x 32 tiles: 64-k).  Kernel
// times (128 x 128 with 16-byte loads, 64 x 64, 32 x 32) of M x N x K:
//   4096 x 4096 x 32    20.6  30.3  67.2    1024 x 1024 x 64   7.9  4.8  6.0
//   4096 x 4096 x 256   79.5  80.6   112    1024 x 1024 x 1000  76  21.6 24.1
//   2392 x 2688 x 8     12.2  16.6  29.5    256 x 256 x 1000    76  19.5  6.9
//   2760 x 960 x 64      9.4   8.8  12.8    800 x 1088 x 8 x 4 batches 8.1 9.3 15.8
// The 128 x 128 kernel holds where C is most of the traffic (a short sum of many
// tiles; 1960 x 1400 x 144 x 17 batches 152, 185, 263) and operands are whole chunks (element loads: 2392 x 2688 x 1 24.9 against 17.1).
enum class TileF32 { k128, k64, k32 };
inline TileF32 tile_f32(uint32_t rows, uint32_t columns, uint32_t inner, uint64_t batches, bool chunked) {
  auto us = [&](uint32_t tile, uint32_t step, double start, double round, double step_us) {
    const double tiles = (double)(((uint64_t)rows + tile - 1) / tile) * (double)(((uint64_t)columns + tile - 1) / tile) * (double)batches;
    return start + std::ceil(tiles / 256) * (round + (double)(((uint64_t)inner + step - 1) / step) * step_us);
  };
  const double us64 = us(64, 32, 3.0, 1.3, 0.45), us32 = us(32, 64, 2.5, 0.75, 0.245);
  if (chunked && inner <= 256 && us(128, 32, 4.5, 2.0, 2.1) < std::fmin(us64, us32)) return TileF32::k128;
  return us32 < us64 ? TileF32::k32 : TileF32::k64;
}

}  // namespace ipus
