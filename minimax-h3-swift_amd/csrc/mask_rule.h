// The mask rules on tile pairs (tile_plan.hip), host and device. Plain C++ as
// well, so a CPU test can compare them with the rules' token-pair definition.
//
// A tile of a lattice rule (LOCAL, AXIAL) past the prefix holds the raster-order
// tokens v0 .. v1 of the video span, so both rules are answered from the tiles'
// ranges instead of from their 128 x 128 token pairs:
//   AXIAL  two tiles share a frame when their frame ranges overlap, and a
//          position when the range of token distances holds a multiple of the
//          frame size (AxialTopology.allows,
//          Sources/H3Attention/AxialTopology.swift:128-137);
//   LOCAL  a tile is a few row segments (frame, y, x0..x1) -- the tile's first
//          and last row and the whole rows between -- and two segments see each
//          other when the frames, the rows' spatial tiles and the ranges of
//          spatial tiles along x are within their windows;
//   both   a key tile that touches a landmark frame is seen by every query, and
//          a tile that touches the prefix sees and is seen by every tile.
#pragma once

#include <cstdint>

#include "../../include/ch3hip.h"

#ifndef __HIPCC__
#ifndef __host__
#define __host__
#define __device__
#endif
#endif

namespace h3hip {

struct RuleDev {
  int32_t kind, seq_len, prefix_len, frames, height, width;
  int32_t frame_window, sp_h, sp_w, sp_window, band;
  int32_t n_tiles;
  const uint8_t* col_global;  // [n_tiles] BAND global columns
  const uint8_t* frame_landmark;  // [frames] landmark flags
};

// Row segments of one tile: 128 with one-token rows, ~128 / width + 2 otherwise.
constexpr int kMaxSegs = H3HIP_TILE;

struct RowSegment {
  int32_t frame, ty, tx0, tx1;  // spatial tile row, first and last spatial tile along x
};

// Video tokens v0 .. v1 of a tile past the prefix, and the lattice rows (counted
// through all frames) they run over.
struct TileSpan {
  int32_t v0, v1, row0, row1;
};

__host__ __device__ inline bool tile_in_prefix(const RuleDev& r, int32_t tile) {
  return tile * H3HIP_TILE < r.prefix_len;
}

__host__ __device__ inline TileSpan tile_span(const RuleDev& r, int32_t tile) {
  const int32_t t0 = tile * H3HIP_TILE;
  const int32_t t1 = t0 + H3HIP_TILE < r.seq_len ? t0 + H3HIP_TILE : r.seq_len;
  const int32_t v0 = t0 - r.prefix_len, v1 = t1 - 1 - r.prefix_len;
  return TileSpan{v0, v1, v0 / r.width, v1 / r.width};
}

// Segment of the span's lattice row `row`, which is row y of frame f.
__host__ __device__ inline RowSegment row_segment(const RuleDev& r, const TileSpan& s,
                                                  int32_t row, int32_t f, int32_t y) {
  const int32_t x0 = row == s.row0 ? s.v0 - row * r.width : 0;
  const int32_t x1 = row == s.row1 ? s.v1 - row * r.width : r.width - 1;
  return RowSegment{f, y / r.sp_h, x0 / r.sp_w, x1 / r.sp_w};
}

__host__ __device__ inline bool ranges_within(int32_t a0, int32_t a1, int32_t b0, int32_t b1,
                                              int32_t window) {
  return a0 - b1 <= window && b0 - a1 <= window;
}

// Whether any token of query tile q sees any token of key tile k under a
// lattice rule, neither tile touching the prefix; seg[0 .. n_seg) are q's row
// segments (LOCAL only).
__host__ __device__ inline bool lattice_tiles_see(const RuleDev& r, const TileSpan& q,
                                                  const TileSpan& k, const RowSegment* seg,
                                                  int32_t n_seg) {
  const int32_t per = r.height * r.width;
  const int32_t kf0 = k.v0 / per, kf1 = k.v1 / per;
  if (r.frame_landmark != nullptr)
    for (int32_t f = kf0; f <= kf1; f++)
      if (r.frame_landmark[f] != 0) return true;
  if (r.kind == H3HIP_RULE_AXIAL) {
    if (ranges_within(q.v0 / per, q.v1 / per, kf0, kf1, 0)) return true;
    // Distances vk - vq run over d0 .. d1: is the largest multiple of the
    // frame size not above d1 at least d0?
    const int32_t d0 = k.v0 - q.v1, d1 = k.v1 - q.v0;
    int32_t m = d1 / per;
    if (d1 < m * per) m--;
    return m * per >= d0;
  }
  int32_t f = kf0, y = k.row0 - f * r.height;
  for (int32_t row = k.row0; row <= k.row1; row++) {
    const RowSegment ks = row_segment(r, k, row, f, y);
    for (int32_t i = 0; i < n_seg; i++) {
      const RowSegment qs = seg[i];
      if (ranges_within(qs.frame, qs.frame, ks.frame, ks.frame, r.frame_window) &&
          ranges_within(qs.ty, qs.ty, ks.ty, ks.ty, r.sp_window) &&
          ranges_within(qs.tx0, qs.tx1, ks.tx0, ks.tx1, r.sp_window))
        return true;
    }
    if (++y == r.height) {
      y = 0;
      f++;
    }
  }
  return false;
}

}  // namespace h3hip
