// Block-sparse flash attention over 128x128 tiles, bf16 MFMA on gfx950.
//
// Persistent workgroups of 8 waves (two per SIMD), one per CU, each running
// the (head, 128-query tile) work units that the plan's XCD-aware schedule
// gives it, one after another; the next unit's first K tile and its Q tile
// load while the current one merges and stores its output. Wave w owns
// queries 32(w&3) .. +31 -- the B operand of v_mfma_f32_32x32x16_bf16 -- and
// key half w>>2 (keys 64(w>>2) .. +63) of every 128-key tile, keeping its own
// online-softmax state; the two key halves of each query are merged exactly
// at the end of the unit.
//
// The tile loop of a unit is one inline-assembly block (bsattn_tile_loop.inc,
// written by gen_tile_loop.py) with every register assigned by hand: O, Q^T
// and a six-entry operand ring in AGPRs (LDS reads land there directly),
// scores and weights double-buffered in VGPRs. In iteration j one instruction
// stream carries the scores of tile j+1, the product with the weights of tile
// j-1, the softmax of tile j and the wave's share of the HBM -> LDS loads of
// K(j+2) and V(j), so each wave's VALU work runs beside its own MFMAs and the
// partner wave on its SIMD fills the issue slots it leaves; one barrier per
// tile orders the loads against the LDS reads.
//
// Each wave computes transposed scores S^T = K Q^T, so a lane holds one
// query's scores and the row max/sum are in-register reductions plus one
// exchange between half-waves. The exponentiated scores are already the B
// operand of O^T = V^T P^T; the A operand V^T is read from the row-major V
// tile with ds_read_b64_tr_b16, whose 16-lane transpose hands lane i column
// c0+i of four consecutive rows.
//
// The softmax is the online recurrence of AxialReference.attendStreamingKeys
// (Sources/H3Attention/AxialReference.swift:129-171) in fp32 and base 2:
// m starts at -3e38 and l and O are rescaled by 2^(m - m_new) when the
// running max moves. Padding keys (>= seq_len, which the reference's unpadded
// arrays do not have) score -inf, not the reference's finite -1e30 mask
// sentinel: their weight is then exactly 0 whatever m is, and a 64-key half
// made only of padding leaves m where it was. (With a finite sentinel that
// half would raise m to round(-1e30 * c), and 2^(-1e30 * c - m) is 2 to the
// power of the product's rounding residual, which can be +1e21: an infinite
// weight times a zeroed V row is NaN.)
// The rescale is lazy: m is only raised when a tile's max exceeds it by more
// than 2^8, which keeps every exponentiated score <= 256 and changes nothing
// in exact arithmetic (numerator and denominator share m). After a row's
// first tile the loop takes the row max only when it may matter: it weighs
// a tile at the current m first, and reruns the full step (max, raise,
// alpha, weights) when the weights of a lane sum past 2^8 or to NaN. l sums the fp32
// weights, as the reference's recurrence does; O accumulates their bf16
// roundings, the P operand of the P V product. The output is O / max(l, 1e-30).
#include <cmath>

#include "bsattn.h"
#include "bsattn_tile_loop.inc"

namespace h3hip {

struct FullLoop {
  static constexpr int kWaves = H3_TILE_LOOP_WAVES, kUnitRows = kTile;
  static __device__ __forceinline__ void run(f32x32& o01, f32x32& o23, float& m, float& l,
                                             const int* ka, const int* va, const int* dk,
                                             const int* dv, int keyoff, int lane16, int rowb,
                                             const LoopScalars& s) {
    asm volatile(H3_TILE_LOOP_ASM
                 : "=&{a[0:31]}"(o01), "=&{a[32:63]}"(o23), "=&{v96}"(m), "=&{v97}"(l)
                 : "{v98}"(ka[0]), "{v99}"(ka[1]), "{v100}"(ka[2]), "{v101}"(ka[3]),
                   "{v102}"(ka[4]), "{v103}"(ka[5]), "{v104}"(ka[6]), "{v105}"(ka[7]),
                   "{v106}"(va[0]), "{v107}"(va[1]), "{v108}"(va[2]), "{v109}"(va[3]),
                   "{v110}"(va[4]), "{v111}"(va[5]), "{v112}"(va[6]), "{v113}"(va[7]),
                   "{v114}"(dk[0]), "{v115}"(dk[1]), "{v116}"(dk[2]), "{v117}"(dk[3]),
                   "{v118}"(dv[0]), "{v119}"(dv[1]), "{v120}"(dv[2]), "{v121}"(dv[3]),
                   "{a120}"(keyoff), "{a121}"(lane16), "{a122}"(rowb),
                   H3_LOOP_SCALARS(s)
                 : H3_TILE_LOOP_CLOBBERS);
  }
};
constexpr int kThreads = 64 * FullLoop::kWaves;
static_assert(FullLoop::kWaves == 8 && H3_TILE_LOOP_ROWS_PER_WAVE == kTile / 8, "tile loop layout");

__global__ __launch_bounds__(kThreads, 1) void bsattn_fwd_kernel(AttnArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t lds[5 * kSlot];
  run_units<FullLoop>(a, lds);
}

// One [heads, rows, 128] view of a caller tensor (strides in elements).
struct View {
  const void* ptr;
  int64_t head_stride, row_stride;
};

static int launch_bsattn(h3hip_plan p, const View& q, const View& k, const View& v,
                         const View& o, int32_t out_rows, float scale, hipStream_t stream) {
  AttnArgs args{static_cast<const uint16_t*>(q.ptr),
                static_cast<const uint16_t*>(k.ptr),
                static_cast<const uint16_t*>(v.ptr),
                static_cast<uint16_t*>(const_cast<void*>(o.ptr)),
                p->d_col_idx,
                p->d_work_ptr,
                p->d_unit_desc,
                q.head_stride,
                k.head_stride,
                v.head_stride,
                o.head_stride,
                (int32_t)q.row_stride,
                (int32_t)k.row_stride,
                (int32_t)v.row_stride,
                (int32_t)o.row_stride,
                p->seq_len,
                out_rows,
                scale * 1.4426950408889634f};
  const unsigned grid = (unsigned)p->groups;
  if (p->work.empty()) return H3HIP_OK;
  if (p->half_units) return launch_bsattn_half(args, grid, stream);
  bsattn_fwd_kernel<<<grid, kThreads, 0, stream>>>(args);
  return check_launch("bsattn_fwd_kernel");
}

// Checks shared by both entry points; H3HIP_OK or the code to return.
static int check_attention_call(h3hip_plan plan, int32_t heads, int32_t head_dim, float scale) {
  H3_REQUIRE(plan != nullptr, H3HIP_EINVAL, "plan is NULL");
  if (head_dim != kD || heads != plan->heads) {
    set_error("declined: head_dim %d heads %d (needs head_dim 128 and the plan's %d heads)",
              head_dim, heads, plan->heads);
    return H3HIP_DECLINED;
  }
  H3_REQUIRE(std::isfinite(scale) && scale > 0.f, H3HIP_EINVAL, "scale must be finite and > 0");
  return H3HIP_OK;
}

}  // namespace h3hip

using namespace h3hip;

extern "C" int h3hip_bsattn_fwd(h3hip_plan plan, const void* q, const void* k, const void* v,
                                int32_t heads, int32_t head_dim, float scale, void* out,
                                int32_t out_layout, void* stream) {
  const int rc = check_attention_call(plan, heads, head_dim, scale);
  if (rc != H3HIP_OK) return rc;
  H3_REQUIRE(q && k && v && out, H3HIP_EINVAL, "NULL tensor argument");
  auto aligned16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  H3_REQUIRE(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out), H3HIP_EINVAL,
             "tensors must be 16-byte aligned");
  H3_REQUIRE(out_layout == H3HIP_OUT_HEAD_MAJOR || out_layout == H3HIP_OUT_TOKEN_MAJOR,
             H3HIP_EINVAL, "unknown out_layout %d", out_layout);
  const int64_t hm = (int64_t)plan->seq_pad * kD;
  const View o = out_layout == H3HIP_OUT_HEAD_MAJOR
                     ? View{out, hm, kD}
                     : View{out, kD, (int64_t)plan->heads * kD};
  return launch_bsattn(plan, View{q, hm, kD}, View{k, hm, kD}, View{v, hm, kD}, o,
                       plan->seq_pad, scale, as_stream(stream));
}

extern "C" int h3hip_bsattn_fwd_strided(h3hip_plan plan, const h3hip_view* q,
                                        const h3hip_view* k, const h3hip_view* v,
                                        int32_t heads, int32_t head_dim, float scale,
                                        const h3hip_view* out, void* stream) {
  const int rc = check_attention_call(plan, heads, head_dim, scale);
  if (rc != H3HIP_OK) return rc;
  H3_REQUIRE(q && k && v && out, H3HIP_EINVAL, "NULL view argument");
  const h3hip_view* views[4] = {q, k, v, out};
  const char* names[4] = {"q", "k", "v", "out"};
  for (int i = 0; i < 4; i++) {
    const h3hip_view& t = *views[i];
    H3_REQUIRE(t.data != nullptr, H3HIP_EINVAL, "%s: NULL data", names[i]);
    H3_REQUIRE((reinterpret_cast<uintptr_t>(t.data) & 15u) == 0, H3HIP_EINVAL,
               "%s: data must be 16-byte aligned", names[i]);
    H3_REQUIRE(t.head_stride >= 0 && t.head_stride % 8 == 0, H3HIP_EINVAL,
               "%s: head_stride %lld must be a non-negative multiple of 8", names[i],
               (long long)t.head_stride);
    H3_REQUIRE(t.row_stride >= kD && t.row_stride % 8 == 0 && t.row_stride <= INT32_MAX,
               H3HIP_EINVAL, "%s: row_stride %lld must be a multiple of 8 and >= %d", names[i],
               (long long)t.row_stride, kD);
  }
  // Q, K and V are fetched with 32-bit offsets from each head's base.
  for (int i = 0; i < 3; i++)
    H3_REQUIRE((int64_t)plan->seq_pad * views[i]->row_stride * 2 < ((int64_t)1 << 31),
               H3HIP_EINVAL, "%s: seq_pad x row_stride exceeds 32-bit offsets", names[i]);
  auto as_view = [](const h3hip_view* t) { return View{t->data, t->head_stride, t->row_stride}; };
  return launch_bsattn(plan, as_view(q), as_view(k), as_view(v), as_view(out), plan->seq_len,
                       scale, as_stream(stream));
}

// The decline policy of H3AttentionBackend.attend (AttentionBackend.swift:123-127)
// with its AttentionContext: H3HIP_OK to run, H3HIP_DECLINED (caller runs
// dense) or an error.
static int attend_policy(h3hip_plan plan, const h3hip_attention_context* ctx) {
  H3_REQUIRE(plan != nullptr, H3HIP_EINVAL, "plan is NULL");
  // No context means dense: a backend that does not know its block or its
  // schedule position cannot honour its own policy
  // (Tests/H3ModulesTests/AttentionSeamTests.swift:127-137).
  if (ctx == nullptr) {
    set_error("declined: no attention context");
    return H3HIP_DECLINED;
  }
  // A plan built for another shape would attend the wrong tiles: refuse the
  // call rather than guess (AxialTopology.swift:65-77).
  if (ctx->sequence_length != plan->seq_len) {
    set_error("declined: sequence length %d, plan built for %d", ctx->sequence_length,
              plan->seq_len);
    return H3HIP_DECLINED;
  }
  if ((plan->kind == H3HIP_RULE_LOCAL || plan->kind == H3HIP_RULE_AXIAL) &&
      ctx->video_start >= 0 &&
      (ctx->video_start != plan->prefix_len || ctx->video_stop != plan->seq_len)) {
    set_error("declined: video span [%d, %d), plan built for [%d, %d)", ctx->video_start,
              ctx->video_stop, plan->prefix_len, plan->seq_len);
    return H3HIP_DECLINED;
  }
  const h3hip_policy& pol = plan->policy;
  if (ctx->block_index < pol.dense_first_blocks ||
      (pol.dense_last_blocks > 0 && ctx->block_index >= ctx->block_count - pol.dense_last_blocks) ||
      ctx->schedule_progress < pol.dense_until_progress ||
      ctx->sequence_length < pol.min_sequence_length) {
    set_error("declined by policy: block %d of %d, progress %.3f", ctx->block_index,
              ctx->block_count, ctx->schedule_progress);
    return H3HIP_DECLINED;
  }
  return H3HIP_OK;
}

extern "C" int h3hip_attend(h3hip_plan plan, const h3hip_attention_context* ctx, const void* q,
                            const void* k, const void* v, int32_t heads, int32_t head_dim,
                            float scale, void* out, void* stream) {
  const int rc = attend_policy(plan, ctx);
  if (rc != H3HIP_OK) return rc;
  return h3hip_bsattn_fwd(plan, q, k, v, heads, head_dim, scale, out, H3HIP_OUT_HEAD_MAJOR,
                          stream);
}

extern "C" int h3hip_attend_strided(h3hip_plan plan, const h3hip_attention_context* ctx,
                                    const h3hip_view* q, const h3hip_view* k,
                                    const h3hip_view* v, int32_t heads, int32_t head_dim,
                                    float scale, const h3hip_view* out, void* stream) {
  const int rc = attend_policy(plan, ctx);
  if (rc != H3HIP_OK) return rc;
  return h3hip_bsattn_fwd_strided(plan, q, k, v, heads, head_dim, scale, out, stream);
}
