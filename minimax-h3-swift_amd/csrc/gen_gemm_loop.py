#!/usr/bin/env python3
"""Writes gemm_loop.inc: the reduction loop of one output tile of
proj_gemm_kernel (proj_gemm.hip) as gfx950 inline assembly, one block per tile
shape, with every register assigned here.

A workgroup of four waves (one per SIMD, two by two) computes 32 NA channels x
32 MB tokens of W x^T; each wave holds NA x MB blocks of
v_mfma_f32_16x16x32_bf16, W rows as A and x rows as B. The reduction runs in
steps of 64, two 32-deep sub-steps each.

  * W and x tiles (rows of 128 bytes a step) go through LDS, in a ring of RW
    and one of RX slots filled by HBM -> LDS loads.
  * A sub-step's NA + MB operands are in registers when it begins; while it
    multiplies, the next sub-step's are read into the other half of the
    operand registers.
  * One barrier per step, between its two sub-steps. Before it a wave has read
    its last operands of step t, so the loads that follow it refill that
    step's slots: x of step t + RX in the step's second sub-step, W of step
    t + RW in the next step's first. It also says that step t + 1's tiles have
    landed, which the second sub-step begins to read.

Every wait is counted: the generator keeps the order in which it issues memory
instructions and waits for exactly the one an instruction needs.

Registers (physical, fixed here):
  a[0 : 4 NA MB - 1]  accumulators, C(na, mb) = a[4 (MB na + mb) : +3]
  v[0 : ..]           operands, A(u, na) and B(u, mb), u = 0, 1
  v[..]               lane offsets (inputs): A and B reads (u, 64 KiB base),
                      x and W loads
  s[64:..]            resources and scalar offsets (clobbered)

Run `python3 gen_gemm_loop.py` in this directory after editing; the generated
file is committed, and tests/test_gemm_loop_gen.py checks it is current and
replays it.
"""
from __future__ import annotations

import os
import sys
from math import lcm

HERE = os.path.dirname(os.path.abspath(__file__))
OUT = os.path.join(HERE, "gemm_loop.inc")

# name (channels x tokens): (NA, MB, RW, RX); 160 KiB of LDS hold the rings
VARIANTS = {"256x256": (8, 8, 3, 2), "256x224": (8, 7, 3, 2), "256x192": (8, 6, 3, 2),
            "256x160": (8, 5, 3, 3), "256x128": (8, 4, 3, 3), "128x192": (4, 6, 4, 4),
            "128x160": (4, 5, 4, 4), "128x128": (4, 4, 5, 5), "128x64": (4, 2, 5, 5)}
WAVES = 4
ROW = 128                 # bytes of a row of one step

# SGPRs
XRS, WRS = "s[64:67]", "s[68:71]"
SJ, SXO, SWO, STMP, SM0 = "s72", "s73", "s74", "s75", "s76"
SGPRS = list(range(64, 77))


class Gen:
    def __init__(self, name):
        self.name = name
        self.na, self.mb, self.rw, self.rx = VARIANTS[name]
        self.w_slot, self.x_slot = 32 * self.na * ROW, 32 * self.mb * ROW
        self.x_at = self.rw * self.w_slot            # x ring after the W ring
        self.lds = self.x_at + self.rx * self.x_slot
        self.w_loads, self.x_loads = self.na, self.mb   # per wave and step, 8 rows each
        ops = self.na + self.mb
        self.unroll = lcm(self.rw, self.rx)
        self.bases = -(-self.lds // 65536)
        at = 8 * ops
        self.ra = at                                 # A read address (base, u)
        self.rb = self.ra + 2 * self.bases
        self.xv = self.rb + 2 * self.bases
        self.wv = self.xv + self.x_loads
        self.n_vgpr = self.wv + self.w_loads
        self.lines = []
        self.issued = []                             # tags of vmem instructions, in order

    def emit(self, *ls):
        self.lines.extend(ls)

    # ---- registers
    def C(self, na, mb):
        b = 4 * (self.mb * na + mb)
        return f"a[{b}:{b + 3}]"

    def A(self, u, na):
        b = 4 * ((self.na + self.mb) * u + na)
        return f"v[{b}:{b + 3}]"

    def B(self, u, mb):
        b = 4 * ((self.na + self.mb) * u + self.na + mb)
        return f"v[{b}:{b + 3}]"

    # ---- memory instructions
    def load(self, which, t, i, step):
        """Rows 8i .. +7 of this wave's share of the W or x tile of step `step`
        into its ring's slot for step t."""
        if which == "x":
            base, m0 = self.x_at + (t % self.rx) * self.x_slot, "%[m0x]"
            v, rs, so = self.xv, XRS, SXO
        else:
            base, m0 = (t % self.rw) * self.w_slot, "%[m0w]"
            v, rs, so = self.wv, WRS, SWO
        g = i % 4
        out = []
        if g == 0:   # one M0 for four loads, whose instruction offsets step both addresses
            out += [f"s_add_u32 m0, {m0}, {base + 1024 * i}", "s_nop 0"]
        out += [f"buffer_load_dwordx4 v{v + i}, {rs}, {so} offen offset:{1024 * g} lds"]
        self.issued.append((which, step))
        return out

    def x_calls(self, t, step):
        return [lambda i=i: self.load("x", t, i, step) for i in range(self.x_loads)]

    def w_calls(self, t, step):
        return [lambda i=i: self.load("w", t, i, step) for i in range(self.w_loads)]

    def wait_for(self, *tags):
        """vmcnt that leaves only what was issued after the last of tags."""
        last = max(i for i, t in enumerate(self.issued) if t in tags)
        return len(self.issued) - 1 - last

    def reads(self, t, u):
        """Operand reads of sub-step (t, u), in the order its MFMAs need them."""
        out = []
        for which, n in (("b", self.mb), ("a", self.na)):
            for k in range(n):
                if which == "a":
                    off, reg, base = (t % self.rw) * self.w_slot, self.A(u, k), self.ra
                else:
                    off, reg, base = self.x_at + (t % self.rx) * self.x_slot, self.B(u, k), self.rb
                b, off = divmod(off + k * 16 * ROW, 65536)
                out.append(f"ds_read_b128 {reg}, v{base + 2 * b + u} offset:{off}")
        return out

    # ---- one step
    def sub_step(self, u, reads, calls):
        """The MFMAs of sub-step u with the next sub-step's operand reads and
        the loads spread between them."""
        n = self.na * self.mb
        reads, calls = list(reads), list(calls)
        nr, nc = len(reads), len(calls)
        done_r = done_c = 0
        if u == 0:   # the wait before the barrier covers sub-step 1's operands
            self.emit("s_waitcnt lgkmcnt(0)")
        for k in range(n):
            na, mb = divmod(k, self.mb)
            c = self.C(na, mb)
            self.emit(f"v_mfma_f32_16x16x32_bf16 {c}, {self.A(u, na)}, {self.B(u, mb)}, {c}")
            # the reads over the first three quarters, so that they are back
            want = min(nr, -(-(k + 1) * nr * 4 // (3 * n)))
            while done_r < want:
                self.emit(reads[done_r])
                done_r += 1
            want = -(-(k + 1) * nc // n)
            while done_c < want:
                self.emit(*calls[done_c]())
                done_c += 1

    def advance(self):
        """Scalar offsets and records of the loads that follow: x of step
        j + RX and W of step j + RW, empty past the last step."""
        self.emit(f"s_add_u32 {SXO}, {SXO}, {ROW}", f"s_add_u32 {SWO}, {SWO}, {ROW}",
                  f"s_add_u32 {STMP}, {SJ}, {self.rx}", f"s_cmp_lt_u32 {STMP}, %[steps]",
                  "s_cselect_b32 s66, s66, 0",
                  f"s_add_u32 {STMP}, {SJ}, {self.rw}", f"s_cmp_lt_u32 {STMP}, %[steps]",
                  "s_cselect_b32 s70, s70, 0")

    def step(self, t, vt, end):
        """Step t (unrolled) traced as step vt, with the exit test at its end."""
        self.sub_step(0, self.reads(t, 1), self.w_calls(t - 1 + self.rw, vt - 1 + self.rw))
        wait = self.wait_for(("w", vt + 1), ("x", vt + 1))
        self.emit(f"s_waitcnt vmcnt({wait}) lgkmcnt(0)", "s_barrier")
        self.advance()
        self.sub_step(1, self.reads(t + 1, 0), self.x_calls(t + self.rx, vt + self.rx))
        self.emit(f"s_add_u32 {SJ}, {SJ}, 1", f"s_cmp_eq_u32 {SJ}, %[steps]",
                  f"s_cbranch_scc1 {end}")
        return wait

    def generate(self):
        em = self.emit
        end, loop = f"L_gemm{self.name}_end_%=", f"L_gemm{self.name}_loop_%="
        em(f"s_mov_b32 {SM0}, m0")
        for i, r in enumerate(("x_lo", "x_hi", "x_rec")):
            em(f"s_mov_b32 s{64 + i}, %[{r}]")
        em("s_mov_b32 s67, 0x20000")
        for i, r in enumerate(("w_lo", "w_hi", "w_rec")):
            em(f"s_mov_b32 s{68 + i}, %[{r}]")
        em("s_mov_b32 s71, 0x20000", f"s_mov_b32 {SJ}, 0")

        def first(which, step):
            off, rec = (SXO, "s66") if which == "x" else (SWO, "s70")
            em(f"s_mov_b32 {off}, {ROW * step}")
            if step:
                em(f"s_cmp_gt_u32 %[steps], {step}", f"s_cselect_b32 {rec}, {rec}, 0")
            for c in (self.x_calls if which == "x" else self.w_calls)(step, step):
                em(*c())
        # The loads before the loop, in the loop's order (x of step t + RX,
        # then W of step t + RW, for t before 0); the loop starts with W of
        # step RW - 1.
        for t in range(-max(self.rw, self.rx), 0):
            if t + self.rx >= 0:
                first("x", t + self.rx)
            if t + self.rw >= 0 and t < -1:
                first("w", t + self.rw)
        s = self.rw - 1
        em(f"s_mov_b32 {SWO}, {ROW * s}", f"s_cmp_gt_u32 %[steps], {s}",
           "s_cselect_b32 s70, s70, 0")
        for r in range(4 * self.na * self.mb):
            em(f"v_accvgpr_write_b32 a{r}, 0")
        em(f"s_waitcnt vmcnt({self.wait_for(('w', 0), ('x', 0))})", "s_barrier")
        em(*self.reads(0, 0))
        em(f"{loop}:")
        waits = [self.step(t, t, end) for t in range(self.unroll)]
        em(f"s_branch {loop}", f"{end}:")
        # The waits of the unrolled steps hold for every later round too.
        later = Gen(self.name)
        later.issued = list(self.issued)
        assert [later.step(t, self.unroll + t, end) for t in range(self.unroll)] == waits
        assert max(waits) < 64
        em("s_waitcnt vmcnt(0) lgkmcnt(0)", "s_barrier", "s_nop 15", "s_nop 15", "s_nop 7",
           f"s_mov_b32 m0, {SM0}")
        return self.lines

    def clobbers(self):
        regs = [f"v{i}" for i in range(self.ra)] + [f"s{i}" for i in SGPRS]
        return regs + ["scc", "memory"]


def render():
    out = ["// Generated by gen_gemm_loop.py -- do not edit; regenerate instead.",
           f"#define H3_GEMM_WAVES {WAVES}"]
    for name, (na, mb, rw, rx) in VARIANTS.items():
        g = Gen(name)
        lines = g.generate()
        body = " \\\n".join('  "' + ln + '\\n"' for ln in lines)
        ins = [f'"{{v{at + i}}}"({arg}[{i}])'
               for arg, at, n in (("RA", g.ra, 2 * g.bases), ("RB", g.rb, 2 * g.bases),
                                  ("XV", g.xv, g.x_loads), ("WV", g.wv, g.w_loads))
               for i in range(n)]
        acc = [f'"=&{{a[{32 * i}:{32 * i + 31}]}}"(C[{i}])' for i in range(-(-na * mb // 8))]
        out += [f"// {32 * na} channels x {32 * mb} tokens: {len(lines)} lines.",
                f"#define H3_GEMM_LDS_{name} {g.lds}",
                f"#define H3_GEMM_BASES_{name} {g.bases}",
                f"#define H3_GEMM_LOOP_{name} \\\n" + body + "\n",
                f"#define H3_GEMM_OUT_{name}(C) " + ", ".join(acc),
                f"#define H3_GEMM_IN_{name}(RA, RB, XV, WV) " + ", ".join(ins),
                f"#define H3_GEMM_CLOBBERS_{name} " + ", ".join(f'"{r}"' for r in g.clobbers())]
    return "\n".join(out) + "\n"


def main():
    text = render()
    if len(sys.argv) > 1 and sys.argv[1] == "--check":
        return 0 if os.path.exists(OUT) and open(OUT).read() == text else 1
    with open(OUT, "w") as f:
        f.write(text)
    return 0


if __name__ == "__main__":
    sys.exit(main())
