// Arguments of the projection kernels (qkv_proj.hip, proj_gemm.hip) and the
// launch of the second.
#pragma once

#include "common.h"
#include "proj_tile.h"

namespace h3hip {

struct ProjArgs {
  const uint16_t* __restrict__ x;        // [seq_len, hidden], row stride ldx
  const uint16_t* __restrict__ w;        // [3 * heads * 128, hidden], row stride ldw
  const uint16_t* __restrict__ q_gamma;  // [128]
  const uint16_t* __restrict__ k_gamma;
  const void* __restrict__ table;        // [seq_len, rot/2, 2, 2]: bf16 (REFERENCE) or fp32
  uint16_t* __restrict__ q_out;          // [heads, seq_pad, 128]
  uint16_t* __restrict__ k_out;
  uint16_t* __restrict__ v_out;
  int64_t ldx, ldw;
  float eps;
  int32_t hidden, rot, seq_len, seq_pad, heads, tiles_m;
  // Out-projection mode: n_out output channels, written token-major into
  // q_out with row stride ldo.
  int32_t n_out;
  int64_t ldo;
  int32_t chunk;   // proj_gemm_kernel: token tiles per chunk of its launch order
};

// 16-byte chunk c of the 128-byte operand row r sits at c ^ ((r >> 1) & 7):
// the 16 rows of a 16-lane read phase cover both row parities x 8 chunk
// positions. Rows 16 apart share the swizzle.
__device__ __forceinline__ int p_swz(int r) { return (r >> 1) & 7; }

// 16-byte chunk c of the 256-byte epilogue row r sits at c ^ e_swz(r): the
// 16 rows one accumulator write covers hit 16 distinct positions (every 8-byte
// slot of a bank window once per 32 lanes), and rows r, r ^ 1 map the chunks
// 0..7 onto complementary halves, so the 2 rows x 8 lanes of a 16-lane read
// phase are conflict-free.
__device__ __forceinline__ int e_swz(int r) { return ((r & 1) << 3) | ((r >> 1) & 7); }

// Launches proj_gemm_kernel on one of its tile shapes (proj_gemm.hip).
int launch_proj_gemm(const ProjArgs& a, ProjTile tile, int32_t rounding, bool plain, bool out,
                     hipStream_t stream);

}  // namespace h3hip
