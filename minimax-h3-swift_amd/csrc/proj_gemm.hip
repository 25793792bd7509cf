// The projections' GEMM on four waves: C = W x^T of h3hip_qkv_proj (with the
// Q/K norm and RoPE in its epilogue, or plain) and of h3hip_out_proj, for every
// size but short reductions that need more than one round of its smaller tiles
// (proj_tile.h).
//
// What bounds it: at random bf16 operands the matrix cores run at the chip's
// power limit, and between them and the operands stands the LDS, which gives
// 128 bytes a clock. Eight waves of 128 x 64 (qkv_proj.hip) read 192 KiB and
// write 64 KiB of LDS a step of 2,048 MFMA cycles, just what it has; four waves
// of 128 x 128 read 128 KiB. One wave per SIMD must then keep its matrix core
// busy alone, so its loop is generated assembly (gen_gemm_loop.py): operands a
// sub-step ahead in registers, the 256 accumulators in AGPRs, every wait
// counted. Measured on MI355X against the eight-wave kernel, in one run: plain
// QKV at 31,885 x 5,120 3.33 against 3.49 ms (1,508 TFLOP/s), with norm and RoPE
// 3.52 against 3.67 ms, out-projection 1.14 against 1.22 ms.
//
// Small grids take smaller tiles of the same loop, so that more CUs work: the
// out-projection of 917 tokens at 5,120 is 80 tiles of 256 x 256 (81 us; 87 on
// eight waves) or 240 of 128 x 160 (42 us), of 300 tokens 40 (80 us) or 200 of 128
// x 64 (25 us). All
// shapes add a channel's products in the same order, so their results are the
// same bits.
//
// Epilogue: the bf16 accumulators go to LDS as token rows (the rings are free
// then), each wave takes whole rows of one head, 8 at a time in the prologue's
// 8-lane layout, and normalises and rotates Q and K with the prologue's device
// code (norm_rope.h) and the render's rotation table. Rows that are complete
// run without a branch so that two passes overlap: one wave per SIMD has no
// other to cover its latencies.
#include <type_traits>

#include "gemm_loop.inc"
#include "norm_rope.h"
#include "proj.h"
#include "tile_order.h"

namespace h3hip {

namespace {

constexpr int kWaves = H3_GEMM_WAVES;
constexpr int kThreads = 64 * kWaves;
constexpr int kHead = 128;
constexpr int kStep = 64;                // reduction per step

typedef float f32x32 __attribute__((ext_vector_type(32)));
// A wave's accumulators, 8 blocks of 16 x 16 to a vector (the last may be part used).
template <int kNA, int kMB>
constexpr int kAccs = (kNA * kMB + 7) / 8;

__device__ __forceinline__ uint32_t uniform(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}

#define H3_SCALARS                                                                          \
  [x_lo] "s"(x_lo), [x_hi] "s"(x_hi), [x_rec] "s"(x_rec), [w_lo] "s"(w_lo), [w_hi] "s"(w_hi), \
      [w_rec] "s"(w_rec), [steps] "s"(steps), [m0x] "s"(m0x), [m0w] "s"(m0w)

// One tile shape: its LDS and its reduction loop, from lane offsets and scalars
// to accumulators.
template <int kNA, int kMB>
struct Shape;
#define H3_SHAPE(NA, MB, NAME)                                                               \
  template <>                                                                                \
  struct Shape<NA, MB> {                                                                     \
    static constexpr int kLds = H3_GEMM_LDS_##NAME, kBases = H3_GEMM_BASES_##NAME;                   \
    static __device__ __forceinline__ void reduce(f32x32 (&c)[kAccs<NA, MB>], const int* ra,   \
                                                  const int* rb, const int* xv, const int* wv, \
                                                  uint32_t x_lo, uint32_t x_hi, uint32_t x_rec, \
                                                  uint32_t w_lo, uint32_t w_hi, uint32_t w_rec, \
                                                  uint32_t steps, uint32_t m0x, uint32_t m0w) { \
      asm volatile(H3_GEMM_LOOP_##NAME                                                       \
                   : H3_GEMM_OUT_##NAME(c)                                                   \
                   : H3_GEMM_IN_##NAME(ra, rb, xv, wv), H3_SCALARS                           \
                   : H3_GEMM_CLOBBERS_##NAME);                                               \
    }                                                                                        \
  };
H3_SHAPE(8, 8, 256x256)
H3_SHAPE(8, 7, 256x224)
H3_SHAPE(8, 6, 256x192)
H3_SHAPE(8, 5, 256x160)
H3_SHAPE(8, 4, 256x128)
H3_SHAPE(4, 6, 128x192)
H3_SHAPE(4, 5, 128x160)
H3_SHAPE(4, 4, 128x128)
H3_SHAPE(4, 2, 128x64)

// The tile's epilogue. Accumulator (na, mb) of lane (g, lr): channels
// 16 (kNA wc + na) + 4g .. +3 of token 16 (kMB wt + mb) + lr. kHl = rot / 16
// (8-channel chunks per rotation half); kPlain: the bf16 GEMM result of every part
// unchanged; kOut: the out-projection, token-major with row stride ldo.
template <int kNA, int kMB, int kMode, int kHl, bool kPlain, bool kOut>
__device__ __forceinline__ void finish_tile(const ProjArgs& a, uint16_t* lds,
                                            const f32x32 (&c)[kAccs<kNA, kMB>], int wave, int lane,
                                            int m0, int n0) {
  constexpr int kTokens = 32 * kMB, kChannels = 32 * kNA;
  const int wc = wave >> 1, wt = wave & 1, lr = lane & 15, g = lane >> 4;
  const int inner = a.heads * kHead;
  // bf16 token rows of the whole tile in LDS; chunk c (16 bytes) of row r sits
  // at c ^ e_swz(r), within its head.
#pragma unroll
  for (int mb = 0; mb < kMB; mb++)
#pragma unroll
    for (int na = 0; na < kNA; na++) {
      const int r = 16 * (kMB * wt + mb) + lr, e = 4 * (kMB * na + mb);
      const f32x32& v = c[e / 32];
      const u32x2 v2 = {cvt_pk(v[e % 32], v[e % 32 + 1]), cvt_pk(v[e % 32 + 2], v[e % 32 + 3])};
      const int chunk = 2 * (kNA * wc + na) + (g >> 1);
      const int pos = (chunk & 16) | ((chunk & 15) ^ e_swz(lr));
      *reinterpret_cast<u32x2*>(lds + r * kChannels + pos * 8 + 4 * (g & 1)) = v2;
    }
  __syncthreads();
  // Each wave takes whole rows of one head: a token half of one of two heads,
  // or a token quarter of a single one.
  constexpr int kHeads = kChannels / kHead, kRows = kTokens * kHeads / kWaves;
  const int nh = kHeads == 2 ? wave >> 1 : 0;
  const int row0 = kRows * (kHeads == 2 ? wave & 1 : wave);
  const int part = kOut ? 0 : n0 / inner;
  const int head = kOut ? 0 : (n0 - part * inner) / kHead + nh;
  uint16_t* out = part == 0 ? a.q_out : part == 1 ? a.k_out : a.v_out;
  const bool norm = !kPlain && !kOut && part < 2;
  constexpr bool kFull = kHl == 8;
  constexpr int kHalf = 8 * kHl;
  const int j = lane & 7, rg = lane >> 3;
  const bool pair_lane = kFull || j < kHl;
  const int chunk_a = pair_lane ? j : 2 * kHl + 2 * (j - kHl);
  const int chunk_b = pair_lane ? j + kHl : chunk_a + 1;
  float gam[16];
  if (norm) {
    const uint16_t* gsrc = part == 0 ? a.q_gamma : a.k_gamma;
    unpack8(*reinterpret_cast<const u32x4*>(gsrc + 8 * chunk_a), gam);
    unpack8(*reinterpret_cast<const u32x4*>(gsrc + 8 * chunk_b), gam + 8);
  }
  // Row r of the tile: this lane's two chunks, normalised and rotated.
  auto finish_row = [&](int r, auto whole, auto rotated) __attribute__((always_inline)) {
    const int m = m0 + r;
    const bool valid = decltype(whole)::value || m < a.seq_len;
    const uint16_t* row = lds + r * kChannels + nh * kHead;
    u32x4 oa = *reinterpret_cast<const u32x4*>(row + ((chunk_a ^ e_swz(r & 15)) * 8));
    u32x4 ob = *reinterpret_cast<const u32x4*>(row + ((chunk_b ^ e_swz(r & 15)) * 8));
    if constexpr (decltype(rotated)::value) {
      RopeEntry tab[8];
      const int64_t entry = (int64_t)(decltype(whole)::value ? m : min(m, a.seq_len - 1)) * kHalf +
                            (pair_lane ? 8 * j : 0);
      if (kMode == H3HIP_ROUND_REFERENCE) {
        const u32x4* tp =
            reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(a.table) + entry * 4);
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const u32x4 tv = tp[q];   // (c, -s, s, c) bf16 of pairs 2q, 2q + 1
          tab[2 * q] = RopeEntry{bf16_lo(tv[0]), bf16_lo(tv[1])};
          tab[2 * q + 1] = RopeEntry{bf16_lo(tv[2]), bf16_lo(tv[3])};
        }
      } else {
        const f32x4* tp = reinterpret_cast<const f32x4*>(a.table) + entry;
#pragma unroll
        for (int e = 0; e < 8; e++) tab[e] = RopeEntry{tp[e][0], tp[e][2]};
      }
      float xr[16];
      unpack8(oa, xr);
      unpack8(ob, xr + 8);
      norm_rope<kMode, kFull>(xr, gam, pair_lane, tab, a.eps, oa, ob);
    }
    if (!valid) oa = ob = u32x4{0u, 0u, 0u, 0u};
    uint16_t* dst = kOut ? a.q_out + (int64_t)m * a.ldo + n0 + nh * kHead
                         : out + ((int64_t)head * a.seq_pad + m) * kHead;
    if (!kOut || valid) {
      *reinterpret_cast<u32x4*>(dst + 8 * chunk_a) = oa;
      *reinterpret_cast<u32x4*>(dst + 8 * chunk_b) = ob;
    }
  };
  // Passes of 8 rows; head-major rows end at seq_pad, a multiple of 8.
  const int passes = kOut ? kRows / 8 : min(kRows, max(a.seq_pad - m0 - row0, 0)) / 8;
  auto finish_rows = [&](auto whole, auto rotated) __attribute__((always_inline)) {
    if constexpr (decltype(whole)::value) {
#pragma unroll 2
      for (int pass = 0; pass < kRows / 8; pass++) finish_row(row0 + 8 * pass + rg, whole, rotated);
    } else {
      for (int pass = 0; pass < passes; pass++) finish_row(row0 + 8 * pass + rg, whole, rotated);
    }
  };
  const bool whole = m0 + row0 + kRows <= a.seq_len;
  if constexpr (!kPlain && !kOut) {
    if (norm) {
      if (whole)
        finish_rows(std::true_type{}, std::true_type{});
      else
        finish_rows(std::false_type{}, std::true_type{});
      return;
    }
  }
  if (whole)
    finish_rows(std::true_type{}, std::false_type{});
  else
    finish_rows(std::false_type{}, std::false_type{});
}

template <int kNA, int kMB, int kMode, int kHl, bool kPlain, bool kOut>
__global__ __launch_bounds__(kThreads, 1) void proj_gemm_kernel(ProjArgs a) {
  using S = Shape<kNA, kMB>;
  constexpr int kTokens = 32 * kMB, kChannels = 32 * kNA;
  __shared__ __attribute__((aligned(16))) uint16_t lds[S::kLds / 2];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wc = wave >> 1, wt = wave & 1;   // channel and token half of the tile
  const int inner = a.heads * kHead;
  const int n_total = kOut ? a.n_out : 3 * inner;
  const TileOrder order{a.tiles_m, n_total / kChannels, a.chunk};
  const int xcd = blockIdx.x % kOrderXcds, slot = blockIdx.x / kOrderXcds;
  if (slot >= order.length(xcd)) return;
  const uint32_t tile = order.tile(xcd, slot);
  const int m0 = (int)(tile >> 16) * kTokens, n0 = (int)(tile & 0xffff) * kChannels;

  const int lr = lane & 15, g = lane >> 4;
  const uint32_t lds_base = uniform((uint32_t)(size_t)(__attribute__((address_space(3))) uint16_t*)lds);
  int ra[2 * S::kBases], rb[2 * S::kBases], xv[kMB], wv[kNA];
#pragma unroll
  for (int b = 0; b < S::kBases; b++)
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int at = (int)lds_base + 65536 * b + (((4 * u + g) ^ p_swz(lr)) * 16);
      ra[2 * b + u] = at + (16 * kNA * wc + lr) * 128;
      rb[2 * b + u] = at + (16 * kMB * wt + lr) * 128;
    }
  const int ldx2 = (int)a.ldx * 2, ldw2 = (int)a.ldw * 2;
  auto load_offset = [&](int rows, int i, int ld2) __attribute__((always_inline)) {
    const int r = rows * wave + 8 * i + (lane >> 3);
    return r * ld2 + (((lane & 7) ^ p_swz(r)) * 16) - 1024 * (i & 3);
  };
#pragma unroll
  for (int i = 0; i < kMB; i++) xv[i] = load_offset(8 * kMB, i, ldx2);
#pragma unroll
  for (int i = 0; i < kNA; i++) wv[i] = load_offset(8 * kNA, i, ldw2);
  const uint64_t xp = (uint64_t)(uintptr_t)(a.x + (int64_t)m0 * a.ldx);
  const uint64_t wp = (uint64_t)(uintptr_t)(a.w + (int64_t)n0 * a.ldw);
  const uint32_t x_lo = uniform((uint32_t)xp), x_hi = uniform((uint32_t)(xp >> 32));
  const uint32_t w_lo = uniform((uint32_t)wp), w_hi = uniform((uint32_t)(wp >> 32));
  const uint32_t x_rec = uniform(m0 < a.seq_len ? (uint32_t)((a.seq_len - 1 - m0) * ldx2 + a.hidden * 2) : 0u);
  const uint32_t w_rec = uniform((uint32_t)(kChannels * ldw2));
  const uint32_t steps = uniform((uint32_t)(a.hidden / kStep));
  const uint32_t m0w = uniform(lds_base + 1024u * kNA * wave);
  const uint32_t m0x = uniform(lds_base + 1024u * kMB * wave);
  f32x32 c[kAccs<kNA, kMB>];
  S::reduce(c, ra, rb, xv, wv, x_lo, x_hi, x_rec, w_lo, w_hi, w_rec, steps, m0x, m0w);

  // The lane again, from the lane counter: kept from before the loop it would
  // be spilled across it.
  int lane2;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane2));
  finish_tile<kNA, kMB, kMode, kHl, kPlain, kOut>(a, lds, c, wave, lane2, m0, n0);
}

template <int kNA, int kMB>
int launch(ProjArgs a, int32_t rounding, bool plain, bool out, hipStream_t st) {
  const ProjGrid g = proj_grid(out ? a.seq_len : a.seq_pad, out ? a.n_out : 3 * a.heads * kHead,
                               32 * kMB, 32 * kNA);
  a.tiles_m = g.order.tiles_m;
  a.chunk = g.order.chunk;
  const dim3 grid(kOrderXcds * g.longest);
  constexpr int kRef = H3HIP_ROUND_REFERENCE, kF32 = H3HIP_ROUND_FP32;
  if (out)
    proj_gemm_kernel<kNA, kMB, kRef, 8, true, true><<<grid, kThreads, 0, st>>>(a);
  else if (plain)
    proj_gemm_kernel<kNA, kMB, kRef, 8, true, false><<<grid, kThreads, 0, st>>>(a);
  else if (rounding == kRef && a.rot == 128)
    proj_gemm_kernel<kNA, kMB, kRef, 8, false, false><<<grid, kThreads, 0, st>>>(a);
  else if (rounding == kRef)
    proj_gemm_kernel<kNA, kMB, kRef, 6, false, false><<<grid, kThreads, 0, st>>>(a);
  else if (a.rot == 128)
    proj_gemm_kernel<kNA, kMB, kF32, 8, false, false><<<grid, kThreads, 0, st>>>(a);
  else
    proj_gemm_kernel<kNA, kMB, kF32, 6, false, false><<<grid, kThreads, 0, st>>>(a);
  return check_launch("proj_gemm_kernel");
}

}  // namespace

int launch_proj_gemm(const ProjArgs& a, ProjTile tile, int32_t rounding, bool plain, bool out,
                     hipStream_t stream) {
  switch (tile) {
    case ProjTile::k256x256: return launch<8, 8>(a, rounding, plain, out, stream);
    case ProjTile::k256x224: return launch<8, 7>(a, rounding, plain, out, stream);
    case ProjTile::k256x192: return launch<8, 6>(a, rounding, plain, out, stream);
    case ProjTile::k256x160: return launch<8, 5>(a, rounding, plain, out, stream);
    case ProjTile::k256x128: return launch<8, 4>(a, rounding, plain, out, stream);
    case ProjTile::k128x192: return launch<4, 6>(a, rounding, plain, out, stream);
    case ProjTile::k128x160: return launch<4, 5>(a, rounding, plain, out, stream);
    case ProjTile::k128x128: return launch<4, 4>(a, rounding, plain, out, stream);
    default: return launch<4, 2>(a, rounding, plain, out, stream);
  }
}

}  // namespace h3hip
