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
  k128x192,
  k128x160,
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
    {ProjTile::k256x192, 256, 192, 0.78}, {ProjTile::k256x160, 256, 160, 0.67},
    {ProjTile::k256x128, 256, 128, 0.57}, {ProjTile::k128x192, 128, 192, 0.50},
    {ProjTile::k128x160, 128, 160, 0.40}, {ProjTile::k128x128, 128, 128, 0.39},
    {ProjTile::k128x64, 128, 64, 0.28},
};

// The launch order of a grid, and how many tiles its longest XCD list gives
// each of that XCD's 32 CUs. Chunks of four token tiles share the most in an
// XCD's L2, but the lists then differ by up to two chunks, which can cost a
// grid that just fits the chip a second round (252 tiles in lists of up to 34);
// smaller chunks are taken when they save a round, and looked at only while the
// lists are not yet as short as they can be: every projection call asks for
// nine grids, and counting all lists of all chunks took 0.9 us of it, this takes 0.15.
struct ProjGrid {
  TileOrder order;
  int longest, rounds;
};
inline ProjGrid proj_grid(int tokens, int channels, int tile_tokens, int tile_channels) {
  const int tiles_m = (tokens + tile_tokens - 1) / tile_tokens, tiles_n = channels / tile_channels;
  const int least = (tiles_m * tiles_n + 32 * kOrderXcds - 1) / (32 * kOrderXcds);
  ProjGrid best{};
  for (int chunk = kOrderChunk; chunk >= 1 && (chunk == kOrderChunk || best.rounds > least);
       chunk /= 2) {
    ProjGrid g{{tiles_m, tiles_n, chunk}, 0, 0};
    g.longest = g.order.longest();
    g.rounds = (g.longest + 31) / 32;
    if (chunk == kOrderChunk || g.rounds < best.rounds) best = g;
  }
  return best;
}

// The tile whose rounds take the least time. A shape's cost is fitted to what
// MI355X measures for it against a 256 x 256 tile's round (0.88-0.97, 0.76-0.93,
// 0.63-0.84, 0.55-0.77, 0.42-0.57, 0.38-0.53, 0.33-0.47 and 0.23-0.35, from a full chip's
// to an almost empty one's), over 64 sizes from 64 to 4,096 tokens of four layers:
// the picks were the fastest shape or within 1.2% of it at 61 of them. Few
// tiles are where it matters: 2,048 tokens x 5,120 channels are 160 tiles of 256
// tokens (87-99 us) or 220 of 192 (80-82 us), 917 tokens 80 tiles (82 us), or 160 of
// 256 x 128 (52 us) or 240 of 128 x 160 (42 us).
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
    const int rounds = proj_grid(tokens, channels, s.tokens, s.channels).rounds;
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
