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
//   LOCAL  a tile is at most five boxes (frames x spatial tile rows x spatial
//          tile columns): its first row, the whole rows to the end of its first
//          frame, the whole frames between, the whole rows of its last frame and
//          its last row; two boxes see each other when their ranges are within
//          the windows along each axis. However narrow the lattice, a pair of
//          tiles is 25 such comparisons at most;
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

// Ranges of frames, spatial tile rows and spatial tile columns, ends included.
struct RuleBox {
  int32_t f0, f1, ty0, ty1, tx0, tx1;
};
constexpr int kMaxBoxes = 5;

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

__host__ __device__ inline bool ranges_within(int32_t a0, int32_t a1, int32_t b0, int32_t b1,
                                              int32_t window) {
  return a0 - b1 <= window && b0 - a1 <= window;
}

__host__ __device__ inline bool boxes_see(const RuleDev& r, const RuleBox& a, const RuleBox& b) {
  return ranges_within(a.f0, a.f1, b.f0, b.f1, r.frame_window) &&
         ranges_within(a.ty0, a.ty1, b.ty0, b.ty1, r.sp_window) &&
         ranges_within(a.tx0, a.tx1, b.tx0, b.tx1, r.sp_window);
}

// The boxes of a tile past the prefix. A tile that lacks one of the five (it ends
// in its first frame, say) repeats its first box in its place.
__host__ __device__ inline void tile_boxes(const RuleDev& r, const TileSpan& s,
                                           RuleBox (&box)[kMaxBoxes]) {
  const int32_t f0 = s.row0 / r.height, f1 = s.row1 / r.height;
  const int32_t y0 = s.row0 - f0 * r.height, y1 = s.row1 - f1 * r.height;
  const int32_t ty0 = y0 / r.sp_h, ty1 = y1 / r.sp_h;
  const int32_t tx0 = (s.v0 - s.row0 * r.width) / r.sp_w;
  const int32_t tx1 = (s.v1 - s.row1 * r.width) / r.sp_w;
  const int32_t last_ty = (r.height - 1) / r.sp_h, last_tx = (r.width - 1) / r.sp_w;
  // (y0 + 1) / sp_h and (y1 - 1) / sp_h
  const int32_t ty_after = ty0 + (y0 + 1 == (ty0 + 1) * r.sp_h ? 1 : 0);
  const int32_t ty_before = ty1 - (y1 == ty1 * r.sp_h ? 1 : 0);
  const bool one_frame = f0 == f1;
  const RuleBox first{f0, f0, ty0, ty0, tx0, s.row0 == s.row1 ? tx1 : last_tx};
  box[0] = first;
  box[1] = one_frame ? y1 - y0 > 1 ? RuleBox{f0, f0, ty_after, ty_before, 0, last_tx} : first
           : y0 + 1 < r.height ? RuleBox{f0, f0, ty_after, last_ty, 0, last_tx} : first;
  box[2] = f1 - f0 > 1 ? RuleBox{f0 + 1, f1 - 1, 0, last_ty, 0, last_tx} : first;
  box[3] = !one_frame && y1 > 0 ? RuleBox{f1, f1, 0, ty_before, 0, last_tx} : first;
  box[4] = s.row1 > s.row0 ? RuleBox{f1, f1, ty1, ty1, 0, tx1} : first;
}

// Whether any token of query tile q sees any token of key tile k under a
// lattice rule, neither tile touching the prefix; box are q's boxes (LOCAL only).
__host__ __device__ inline bool lattice_tiles_see(const RuleDev& r, const TileSpan& q,
                                                  const TileSpan& k,
                                                  const RuleBox (&box)[kMaxBoxes]) {
  const int32_t kf0 = k.row0 / r.height, kf1 = k.row1 / r.height;
  if (r.kind == H3HIP_RULE_AXIAL) {
    const int32_t per = r.height * r.width;
    if (ranges_within(q.row0 / r.height, q.row1 / r.height, kf0, kf1, 0)) return true;
    // Distances vk - vq run over d0 .. d1: is the largest multiple of the
    // frame size not above d1 at least d0?
    const int32_t d0 = k.v0 - q.v1, d1 = k.v1 - q.v0;
    int32_t m = d1 / per;
    if (d1 < m * per) m--;
    if (m * per >= d0) return true;
  } else {
    RuleBox kb[kMaxBoxes];
    tile_boxes(r, k, kb);
    bool hit = false;
    for (const RuleBox& a : box)
      for (const RuleBox& b : kb) hit |= boxes_see(r, a, b);
    if (hit) return true;
  }
  // Up to 128 flags where a frame is one token, read without waiting for each
  // other.
  bool landmark = false;
  if (r.frame_landmark != nullptr)
    for (int32_t f = kf0; f <= kf1; f++) landmark |= r.frame_landmark[f] != 0;
  return landmark;
}

}  // namespace h3hip
