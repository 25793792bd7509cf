// What the two attention kernels share: their arguments, the LDS layout, the
// loads that start a unit, and the persistent unit loop around the generated
// tile loop. bsattn_fwd.hip runs it on eight waves with units of 128 queries,
// bsattn_half.hip on four with units of 64.
#pragma once

#include <type_traits>

#include "common.h"
#include "plan.h"

namespace h3hip {

constexpr int kTile = 128;
constexpr int kD = 128;
constexpr int kSlot = kTile * kD;                   // one K or V tile, unpadded (elements)
// LDS byte layout: K slots 0 and 1, V slots 0 and 1, the unit's Q tile.
constexpr uint32_t kKSlot0 = 0, kVSlot0 = 65536, kQSlot = 131072;
// s_waitcnt immediate for vmcnt(0) with expcnt and lgkmcnt left unconstrained
// (gfx9 encoding: vmcnt[3:0] bits 3:0, expcnt bits 6:4, lgkmcnt bits 11:8,
// vmcnt[5:4] bits 15:14).
constexpr int kWaitVmcnt0 = 0x0F70;
// Buffer resource word 3 for raw (untyped, unswizzled) buffer loads on gfx9:
// DATA_FORMAT = 32 bits, everything else zero.
constexpr int kBufferWord3 = 0x00020000;

// Each tensor is a [heads, rows, 128] view: element (h, s, d) at
// base + h*head_stride + s*row_stride + d. Only rows < seq_len of q, k and v
// are read; rows < out_rows of out are written (zero past seq_len).
struct AttnArgs {
  const uint16_t* __restrict__ q;
  const uint16_t* __restrict__ k;
  const uint16_t* __restrict__ v;
  uint16_t* __restrict__ out;
  const int32_t* __restrict__ col_idx;
  const int32_t* __restrict__ work_ptr;  // [groups + 1]
  const int32_t* __restrict__ unit_desc;  // [units][kUnitDescInts], in work order
  int64_t q_hs, k_hs, v_hs, o_hs;  // head strides (elements)
  int32_t q_rs, k_rs, v_rs, o_rs;  // row strides (elements)
  int32_t seq_len, out_rows;
  float scale_log2;
};

typedef __attribute__((address_space(3))) void lds_void;
typedef float f32x32 __attribute__((ext_vector_type(32)));

// LDS tiles are unpadded 256-byte rows whose 16-byte chunks are XOR-swizzled
// so the operand reads hit 64 distinct banks per phase:
//   K and Q: chunk c of row r sits at c ^ (r & 15) -- 16 consecutive rows read
//      at one chunk (ds_read_b128) land on 16 different chunk positions;
//   V: chunk c of row r sits at c ^ (4*(r & 3) + ((r >> 2) & 3)) -- the
//      transpose load reads 4 consecutive rows x 4 consecutive chunks per
//      32-lane phase, which this maps onto all 16 chunk positions.
__host__ __device__ __forceinline__ int k_swz(int r) { return r & 15; }
__host__ __device__ __forceinline__ int v_swz(int r) { return 4 * (r & 3) + ((r >> 2) & 3); }

// Workgroup barrier ordering this wave's LDS accesses only (not its
// outstanding global loads and stores, which __syncthreads would also wait for).
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

// A unit's first K tile and its Q rows, HBM -> LDS: wave w moves its share of
// the rows of each, 4 rows per instruction, chunks K-swizzled, into K slot 0 and
// the Q slot. Buffer resources bound the rows
// at seq_len, so no row past it is fetched; query rows past it only feed
// output rows that are stored as zeros.
// Unit iu's descriptor (plan.h: unit, col_idx index, n, c0, c1, c2, ragged),
// through the scalar cache.
__device__ __forceinline__ const __attribute__((address_space(4))) int32_t* unit_desc(
    const AttnArgs& a, int iu) {
  return (const __attribute__((address_space(4))) int32_t*)(a.unit_desc) + kUnitDescInts * iu;
}

// First query row of the unit within its q-tile (half units only).
template <class Loop>
__device__ __forceinline__ int unit_row0(const __attribute__((address_space(4))) int32_t* desc) {
  return Loop::kUnitRows == kTile ? 0 : desc[7];
}

template <class Loop>
__device__ __forceinline__ void load_unit_start(const AttnArgs& a, uint16_t* lds, int iu,
                                                int wave, int lane) {
  const auto* d = unit_desc(a, iu);
  const int32_t unit = d[0];
  const int head = unit >> 16, qt = unit & 0xffff;
  auto tile = [&](const uint16_t* base, int rs2, int row0, uint16_t* slot, auto rows)
      __attribute__((always_inline)) {
    constexpr int kRows = decltype(rows)::value;   // this wave's
    const int dma_row = kRows * wave + (lane >> 4);
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)base, 0, (a.seq_len - 1) * rs2 + kD * 2, kBufferWord3);
#pragma unroll
    for (int i = 0; i < kRows / 4; i++) {
      const int row = dma_row + 4 * i;
      const int voff = (row0 + row) * rs2 + (((lane & 15) ^ k_swz(row)) * 16);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc, (lds_void*)(slot + (kRows * wave + 4 * i) * kD), 16, voff, 0, 0, 0);
    }
  };
  tile(a.q + head * a.q_hs, a.q_rs * 2, qt * kTile + unit_row0<Loop>(d), lds + kQSlot / 2,
       std::integral_constant<int, Loop::kUnitRows / Loop::kWaves>{});
  if (d[2] > 0)
    tile(a.k + head * a.k_hs, a.k_rs * 2, d[3] * kTile, lds + kKSlot0 / 2,
         std::integral_constant<int, kTile / Loop::kWaves>{});
}

// Wave-uniform inputs of a tile loop.
struct LoopScalars {
  uint32_t n, c0, c1, c2, colp_lo, colp_hi, kb_lo, kb_hi, vb_lo, vb_hi, krec, vrec, kstep, vstep,
      c, m0k, m0v, qoff, seq, ragged;
};
#define H3_LOOP_SCALARS(S)                                                                    \
  [n] "s"(S.n), [c0] "s"(S.c0), [c1] "s"(S.c1), [c2] "s"(S.c2), [colp_lo] "s"(S.colp_lo),     \
      [colp_hi] "s"(S.colp_hi), [kb_lo] "s"(S.kb_lo), [kb_hi] "s"(S.kb_hi),                   \
      [vb_lo] "s"(S.vb_lo), [vb_hi] "s"(S.vb_hi), [krec] "s"(S.krec), [vrec] "s"(S.vrec),     \
      [kstep] "s"(S.kstep), [vstep] "s"(S.vstep), [c] "s"(S.c), [m0k] "s"(S.m0k),             \
      [m0v] "s"(S.m0v), [qoff] "s"(S.qoff), [seq] "s"(S.seq), [ragged] "s"(S.ragged)

// A workgroup's units. Loop: kWaves, kUnitRows (queries of a unit) and run(),
// the generated tile loop. Wave w owns queries 32 (w % kGroups) .. +31 of the unit
// and key half w / kGroups.
template <class Loop>
__device__ __forceinline__ void run_units(const AttnArgs& a, uint16_t* lds) {
  constexpr int kGroups = Loop::kUnitRows / 32, kRowsPerWave = kTile / Loop::kWaves;
  constexpr int kLoads = kRowsPerWave / 4;
  static_assert(2 * kGroups == Loop::kWaves, "query groups x key halves");

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform, in an SGPR
  const int qg = wave % kGroups, kh = wave / kGroups;
  const int k_rs2 = a.k_rs * 2, v_rs2 = a.v_rs * 2;
  const uint32_t base = lds_addr(lds);

  const int u_beg = a.work_ptr[blockIdx.x], u_end = a.work_ptr[blockIdx.x + 1];
  if (u_beg < u_end) load_unit_start<Loop>(a, lds, u_beg, wave, threadIdx.x & 63);
  // Lane address offsets of the tile loop (bytes), the same for every unit:
  // computed once; the tile loop takes them as inputs and leaves them intact.
  const int lane0 = threadIdx.x & 63, li0 = lane0 & 31, hh0 = lane0 >> 5;
  int ka[8], va[8], dk[kLoads], dv[kLoads];
#pragma unroll
  for (int s = 0; s < 8; s++)
    ka[s] = base + kKSlot0 + 2 * ((kh * 64 + li0) * kD + (((2 * s + hh0) ^ k_swz(li0)) * 8));
  const int g = lane0 >> 4, mm = lane0 & 15;
#pragma unroll
  for (int p = 0; p < 2; p++)
#pragma unroll
    for (int db = 0; db < 4; db++) {
      const int row = kh * 64 + 8 * p + 4 * (g >> 1) + (mm >> 2);
      const int chunk = 4 * db + 2 * (g & 1) + ((mm & 3) >> 1);
      va[4 * p + db] =
          base + kVSlot0 + 2 * (row * kD + ((chunk ^ v_swz(row)) * 8) + 4 * (mm & 1));
    }
#pragma unroll
  for (int i = 0; i < kLoads; i++) {
    const int row = kRowsPerWave * wave + 4 * i + (lane0 >> 4);
    // Less 1024 (i & 3): the tile loop's loads add it back as their
    // instruction offset, which also steps their LDS address.
    dk[i] = row * k_rs2 + (((lane0 & 15) ^ k_swz(row)) * 16) - 1024 * (i & 3);
    dv[i] = row * v_rs2 + (((lane0 & 15) ^ v_swz(row)) * 16) - 1024 * (i & 3);
  }
  // The first unit's K(0) and Q have landed (later units wait in the merge).
  __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
  for (int iu = u_beg; iu < u_end; iu++) {
    // Lane-derived values are rebuilt for each unit from an opaque copy of the
    // thread index: hoisted out of the unit loop they would stay live across
    // the tile loop, which leaves no VGPRs to hold them.
    int tid;
    asm volatile("v_mov_b32 %0, %1" : "=v"(tid) : "v"(threadIdx.x));
    const int lane = tid & 63, hh = lane >> 5;
    const auto* desc = unit_desc(a, iu);
    const int32_t unit = desc[0];
    const int head = unit >> 16, qt = unit & 0xffff;
    const int q0 = qt * kTile + unit_row0<Loop>(desc) + qg * 32;
    const int beg = desc[1], n = desc[2];

    // The unit's K(0) and Q have landed (each wave waited for its own loads
    // before its output stores) and the previous unit's merge buffers have
    // been read. The output stores stay in flight: loads return in order, so
    // the tile loop's counted waits only grow stronger for them.
    lds_barrier();

    f32x32 o01, o23;  // O(0), O(1) and O(2), O(3): 16 accumulators each
    float m, l;
    if (n > 0) {

      const int keyoff = kh * 64 + 4 * hh, lane16 = 16 * lane;
      const int rowb = kRowsPerWave * wave + (lane >> 4);

      // Scalar operands of the tile loop, made wave-uniform explicitly so they
      // are SGPRs.
      auto u = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };
      const uint32_t c0 = u(desc[3]), c1 = u(desc[4]), c2 = u(desc[5]), ragged = u(desc[6]);
      const uint64_t colp = (uint64_t)(uintptr_t)(a.col_idx + beg);
      const uint64_t kbp = (uint64_t)(uintptr_t)(a.k + head * a.k_hs);
      const uint64_t vbp = (uint64_t)(uintptr_t)(a.v + head * a.v_hs);
      const uint32_t krec = u((uint32_t)((a.seq_len - 1) * k_rs2 + kD * 2));
      const uint32_t vrec = u((uint32_t)((a.seq_len - 1) * v_rs2 + kD * 2));
      const uint32_t m0k = u(base + kKSlot0 + 256u * kRowsPerWave * wave);
      const uint32_t m0v = u(base + kVSlot0 + 256u * kRowsPerWave * wave);
      const uint32_t qoff = u(kQSlot - kKSlot0 + 256u * 32u * qg - 256u * 64u * kh);
      const uint32_t nn = u(n), seq = u(a.seq_len), k128 = u(k_rs2 * kTile), v128 = u(v_rs2 * kTile);
      const uint32_t cbits = u(__float_as_uint(a.scale_log2));
      Loop::run(o01, o23, m, l, ka, va, dk, dv, keyoff, lane16, rowb,
                LoopScalars{nn, c0, c1, c2, u((uint32_t)colp), u((uint32_t)(colp >> 32)),
                            u((uint32_t)kbp), u((uint32_t)(kbp >> 32)), u((uint32_t)vbp),
                            u((uint32_t)(vbp >> 32)), krec, vrec, k128, v128, cbits, m0k, m0v,
                            qoff, seq, ragged});
    } else {
      // A row with no active tile: its output is zero.
      o01 = f32x32{};
      o23 = f32x32{};
      m = -3.0e38f;
      l = 0.f;
    }

    // Lane values again, from a fresh opaque copy: kept from before the tile
    // loop they would be spilled across it.
    asm volatile("v_mov_b32 %0, %1" : "=v"(tid) : "v"(threadIdx.x));
    const int lane2 = tid & 63, li2 = lane2 & 31, hh2 = lane2 >> 5;
    // The next unit's K(0) and Q go into K slot 0 and the Q slot, which no
    // wave reads once its tile loop has passed the last tile's barrier.
    if (iu + 1 < u_end) load_unit_start<Loop>(a, lds, iu + 1, wave, lane2);
    // Every wave's last V reads are done: the V slots are free. An LDS-only
    // barrier: __syncthreads would also wait for the loads just issued, whose
    // HBM latency the merge is there to cover (the next unit waits for them).
    lds_barrier();

    // Merge of the two key halves (exact: both rescaled to the larger m).
    // Wave (qg, kh) finalises channel blocks 2kh, 2kh+1 of its 32 queries and
    // hands the partner wave (qg, 1-kh) its O of the partner's blocks, 8 KiB
    // per wave in V slot 0, with m and l in K slot 1.
    // l summed with the other half-wave's (the same queries' other 32 keys).
    const auto lsw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l),
                                                      false, false);
    const float lt = __uint_as_float(lsw[0]) + __uint_as_float(lsw[1]);
    float* xo = reinterpret_cast<float*>(lds + kVSlot0 / 2);
    float* xml = reinterpret_cast<float*>(lds + kSlot);
    // The wave keeps channel blocks 2kh, 2kh+1 (keep) and gives the other
    // two (give); block 2i + b is register 16b + r of o01 (i = 0) or o23.
    auto merge = [&](const f32x32& keep, const f32x32& give, int kb0)
                     __attribute__((always_inline)) {
      float* mine = xo + wave * 2048;
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r4 = 0; r4 < 4; r4++) {
          const int r = 16 * i + 4 * r4;
          const f32x4 w = {give[r], give[r + 1], give[r + 2], give[r + 3]};
          *reinterpret_cast<f32x4*>(mine + ((4 * i + r4) * 64 + lane2) * 4) = w;
        }
      xml[wave * 128 + lane2] = m;
      xml[wave * 128 + 64 + lane2] = lt;
      lds_barrier();
      const int pw = wave ^ kGroups;
      const float* theirs = xo + pw * 2048;
      const float mp = xml[pw * 128 + lane2], ltp = xml[pw * 128 + 64 + lane2];
      const float mmax = fmaxf(m, mp);
      const float f0 = __builtin_amdgcn_exp2f(m - mmax), f1 = __builtin_amdgcn_exp2f(mp - mmax);
      const float inv = 1.0f / fmaxf(lt * f0 + ltp * f1, 1.0e-30f);
      const float s0 = f0 * inv, s1 = f1 * inv;
      // O^T C layout: lane (li, hh) holds query q0 + li, channels
      // 32db + 8gg + 4hh + [0, 4) in registers 16db + 4gg .. +3.
      const int qi = q0 + li2;
      const bool valid = qi < a.seq_len;
      // This wave's loads of the next unit are done before its output
      // stores are issued, so that the next unit waits for no store.
      __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
      if (qi < a.out_rows) {
        uint16_t* orow = a.out + head * a.o_hs + (int64_t)qi * a.o_rs;
#pragma unroll
        for (int i = 0; i < 2; i++) {
          const int db = kb0 + i;
#pragma unroll
          for (int gg = 0; gg < 4; gg++) {
            const f32x4 t =
                *reinterpret_cast<const f32x4*>(theirs + ((4 * i + gg) * 64 + lane2) * 4);
            float ov[4];
#pragma unroll
            for (int e = 0; e < 4; e++) ov[e] = keep[16 * i + 4 * gg + e] * s0 + t[e] * s1;
            u32x2 w = {0u, 0u};
            if (valid) {
              w[0] = pack_bf16x2(ov[0], ov[1]);
              w[1] = pack_bf16x2(ov[2], ov[3]);
            }
            *reinterpret_cast<u32x2*>(orow + 32 * db + 8 * gg + 4 * hh2) = w;
          }
        }
      }
    };
    if (kh == 0)
      merge(o01, o23, 0);
    else
      merge(o23, o01, 2);
  }
}

// Launches bsattn_half_kernel (bsattn_half.hip) for a plan of half units.
int launch_bsattn_half(const AttnArgs& args, unsigned groups, hipStream_t stream);

}  // namespace h3hip
