// Attention on half units: the unit loop of bsattn_fwd.hip on workgroups of four
// waves and work units of 64 queries, for plans whose units are too few or too
// uneven to keep the CUs busy (plan creation decides, tile_plan.hip).
//
// A launch of few units is bound by one unit's serial chain: its tiles, each
// with its loads' and LDS's latency, and its merge. Half a unit has a shorter
// chain (the LDS gives it its 128 KiB of operand reads a tile in half the time;
// the loads are the same), and there are twice as many. On an idle MI355X it takes
// 0.80 us a tile against 1.07, and 5.4 us against 7.0 beyond its tiles, launch
// included; where all CUs work, two half units take 1.13-1.28 times a whole one's
// time. Measured, full against half units: a band of 4,096 tokens x 4 heads 14.1 ->
// 11.1 us, 917 dense tokens x 8 heads 15.6-16.3 -> 11.7-12.2 us, 5,372 x 2 heads 52.1-53.4
// -> 40.4-41.7 us, and 31,885 local tokens x 2 heads, whose few prefix rows see every
// tile, 290-295 -> 234-237 us. Each query's arithmetic is the same, in the same
// order: so are the bits. One wave per SIMD leaves the registers for eight loads
// a tile; the tile loop is generated (gen_half_loop.py).
#include "bsattn.h"
#include "bsattn_half_loop.inc"

namespace h3hip {

namespace {

struct HalfLoop {
  static constexpr int kWaves = H3_HALF_LOOP_WAVES, kUnitRows = kTile / 2;
  static __device__ __forceinline__ void run(f32x32& o01, f32x32& o23, float& m, float& l,
                                             const int* ka, const int* va, const int* dk,
                                             const int* dv, int keyoff, int lane16, int rowb,
                                             const LoopScalars& s) {
    asm volatile(H3_HALF_LOOP_ASM
                 : "=&{a[0:31]}"(o01), "=&{a[32:63]}"(o23), "=&{v96}"(m), "=&{v97}"(l)
                 : "{v98}"(ka[0]), "{v99}"(ka[1]), "{v100}"(ka[2]), "{v101}"(ka[3]), "{v102}"(ka[4]), "{v103}"(ka[5]), "{v104}"(ka[6]), "{v105}"(ka[7]),
                   "{v106}"(va[0]), "{v107}"(va[1]), "{v108}"(va[2]), "{v109}"(va[3]), "{v110}"(va[4]), "{v111}"(va[5]), "{v112}"(va[6]), "{v113}"(va[7]),
                   "{v114}"(dk[0]), "{v115}"(dk[1]), "{v116}"(dk[2]), "{v117}"(dk[3]), "{v118}"(dk[4]), "{v119}"(dk[5]), "{v120}"(dk[6]), "{v121}"(dk[7]),
                   "{v122}"(dv[0]), "{v123}"(dv[1]), "{v124}"(dv[2]), "{v125}"(dv[3]), "{v126}"(dv[4]), "{v127}"(dv[5]), "{v128}"(dv[6]), "{v129}"(dv[7]),
                   "{a120}"(keyoff), "{a121}"(lane16), "{a122}"(rowb), H3_LOOP_SCALARS(s)
                 : H3_HALF_LOOP_CLOBBERS);
  }
};
constexpr int kThreads = 64 * HalfLoop::kWaves;
static_assert(HalfLoop::kWaves == 4 && H3_HALF_LOOP_ROWS_PER_WAVE == kTile / 4, "tile loop layout");

__global__ __launch_bounds__(kThreads, 1) void bsattn_half_kernel(AttnArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t lds[5 * kSlot];
  run_units<HalfLoop>(a, lds);
}

}  // namespace

int launch_bsattn_half(const AttnArgs& args, unsigned groups, hipStream_t stream) {
  bsattn_half_kernel<<<groups, kThreads, 0, stream>>>(args);
  return check_launch("bsattn_half_kernel");
}

}  // namespace h3hip
