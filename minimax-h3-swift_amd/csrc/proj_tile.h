// Which kernel and tile shape a projection of these sizes runs on. Plain C++,
// so a CPU test can check it.
#pragma once

#include <algorithm>

#include "tile_order.h"

namespace h3hip {

enum class ProjTile {
  kEightWave,   // qkv_proj_kernel, 256 channels x 256 tokens
  k256x256,     // proj_gemm_kernel, channels x tokens
  k256x224,
  k256x192,
  k256x160,
  k256x128,
  k128x128,
  k128x64,
};

struct ProjShape {
  ProjTile tile;
  int channels, tokens;
  double cost;   // time of a tile where all CUs are busy, that of 256 x 256 being 1
};
constexpr ProjShape kProjShapes[] = {
    {ProjTile::k256x256, 256, 256, 1.00}, {ProjTile::k256x224, 256, 224, 0.90},
    {ProjTile::k256x192, 256, 192, 0.78}, {ProjTile::k256x160, 256, 160, 0.68},
    {ProjTile::k256x128, 256, 128, 0.57}, {ProjTile::k128x128, 128, 128, 0.36},
    {ProjTile::k128x64, 128, 64, 0.30},
};

// Tiles the longest XCD list gives each of its 32 CUs.
inline int proj_rounds(int tokens, int channels, int tile_tokens, int tile_channels) {
  const TileOrder order{(tokens + tile_tokens - 1) / tile_tokens, channels / tile_channels};
  int longest = 0;
  for (int x = 0; x < kOrderXcds; x++) longest = std::max(longest, order.length(x));
  return (longest + 31) / 32;
}

// The tile whose rounds take the least time. A shape's cost is what MI355X
// measures for it where all CUs are busy (0.88-0.92, 0.76-0.80, 0.66-0.70,
// 0.56-0.60, 0.35-0.40 and 0.28-0.31 of a 256 x 256 tile over 22 token counts from 64 to
// 18,102 and four layers); the picks were the fastest shape, or within 1.5% of
// it, at 87 of those 88 sizes. Few tiles are where it matters: 2,048 tokens x
// 5,120 channels are 160 tiles of 256 tokens (90 us) or 220 of 192 (80 us).
//
// With few reduction steps a tile is mostly its fill and epilogue: there the
// eight-wave kernel, whose two waves per SIMD cover each other's epilogue, is
// the faster one (18,102 tokens x 40 heads at hidden 512: 361 against 382 us with
// norm and RoPE, 289 against 295 us plain; equal at about 1,024 plain and 1,536
// with them), and other tiles pay only while they need one round and save a
// third (224 and 192 tokens were 3-10% slower than it at hidden 64-512).
inline ProjTile pick_proj_tile(int tokens, int channels, int hidden, bool fused) {
  const bool few_steps = hidden < (fused ? 1536 : 1024);
  double best = 0;
  ProjTile tile = ProjTile::kEightWave;
  for (const ProjShape& s : kProjShapes) {
    const int rounds = proj_rounds(tokens, channels, s.tokens, s.channels);
    const double cost = s.cost * rounds;
    if (s.tile == ProjTile::k256x256) {
      best = cost;
      if (!few_steps) tile = s.tile;
    } else if (cost < best && !(few_steps && (rounds > 1 || s.cost > 0.7))) {
      best = cost;
      tile = s.tile;
    }
  }
  return tile;
}

}  // namespace h3hip
