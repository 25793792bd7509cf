// Which kernel and tile shape a projection of these sizes runs on. Plain C++,
// so a CPU test can check it.
#pragma once

#include <algorithm>

#include "tile_order.h"

namespace h3hip {

enum class ProjTile {
  kEightWave,   // qkv_proj_kernel, 256 channels x 256 tokens
  k256x256,     // proj_gemm_kernel, channels x tokens
  k256x128,
  k128x128,
};

// Tiles the longest XCD list gives each of its 32 CUs.
inline int proj_rounds(int tokens, int channels, int tile_tokens, int tile_channels) {
  const TileOrder order{(tokens + tile_tokens - 1) / tile_tokens, channels / tile_channels};
  int longest = 0;
  for (int x = 0; x < kOrderXcds; x++) longest = std::max(longest, order.length(x));
  return (longest + 31) / 32;
}

// A tile of 256 x 128 takes 0.58 and one of 128 x 128 0.37 of the time of a
// 256 x 256 tile where all CUs are busy (MI355X, hidden 5,120 and 5,376: 0.55-0.57 and
// 0.35-0.38), so the larger tile is the faster one unless the last round of
// the smaller ones fills the chip better. With few reduction steps a tile is
// mostly its fill and epilogue: there the eight-wave kernel, whose two waves
// per SIMD cover each other's epilogue, is the faster one (41,600 tokens-heads
// at hidden 512: 361 against 382 us fused, 289 against 295 us plain; equal at
// about 1,024 plain and 1,536 fused), and smaller tiles only pay while they
// need one round.
inline ProjTile pick_proj_tile(int tokens, int channels, int hidden, bool fused) {
  const bool few_steps = hidden < (fused ? 1536 : 1024);
  const int r256 = proj_rounds(tokens, channels, 256, 256);
  const int r128t = proj_rounds(tokens, channels, 128, 256);
  const int r128 = proj_rounds(tokens, channels, 128, 128);
  double best = r256;
  ProjTile tile = few_steps ? ProjTile::kEightWave : ProjTile::k256x256;
  if (0.58 * r128t < best && !(few_steps && r128t > 1)) {
    best = 0.58 * r128t;
    tile = ProjTile::k256x128;
  }
  if (0.37 * r128 < best && !(few_steps && r128 > 1)) tile = ProjTile::k128x128;
  return tile;
}

}  // namespace h3hip
