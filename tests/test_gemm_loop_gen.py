"""The generated reduction loop of proj_gemm_kernel (csrc/gen_gemm_loop.py ->
csrc/gemm_loop.inc), replayed on the CPU instruction by instruction.

The replay runs the scalar code (so every branch, scalar offset and record
count is the one the GPU would take) and follows which rows and which step each
LDS piece, operand register and accumulator holds, for all four waves of the
workgroup, which run the same stream. A load has landed once a counted vmcnt
wait covers it; another wave's load only once a barrier follows that wait. It
fails when

  * an operand read touches a piece that has not landed in every wave or holds
    another step;
  * a load refills a piece that some wave may still have to read;
  * an MFMA reads an operand still in flight, or not the step it belongs to;
  * an accumulator does not add up every sub-step of every step once, in order;
  * a load past the last step is not empty.

Each of these is also planted once and must be found."""
import importlib.util
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "minimax-h3-swift_amd", "csrc")
spec = importlib.util.spec_from_file_location("gen_gemm_loop",
                                              os.path.join(CSRC, "gen_gemm_loop.py"))
G = importlib.util.module_from_spec(spec)
spec.loader.exec_module(G)


class Wrong(AssertionError):
    pass


def check(cond, *what):
    if not cond:
        raise Wrong(what)


def _span(tok):
    m = re.match(r"[va]\[(\d+):(\d+)\]", tok)
    return tuple(range(int(m.group(1)), int(m.group(2)) + 1))


def replay(g, lines, steps):
    """Runs the stream; returns what each accumulator summed, in order."""
    labels = {ln[:-1]: i for i, ln in enumerate(lines) if ln.endswith(":")}
    ins = {"%[steps]": steps, "%[m0w]": 0, "%[m0x]": 0, "%[x_lo]": 0, "%[x_hi]": 0,
           "%[w_lo]": 0, "%[w_hi]": 0, "%[x_rec]": 1, "%[w_rec]": 1, "m0": 0}
    s, scc = dict(ins), False
    tile = {"w": (0, 32 * g.na // 8), "x": (g.x_at, 32 * g.mb // 8)}   # first byte, pieces
    per_wave = {"w": g.na, "x": g.mb}
    piece = {}          # address / 1024 -> (which, step, index), the load's number, its barrier
    free_after = {}     # address / 1024 -> barriers passed when its last read returned
    vm, landed, lgkm = [], 0, []       # loads in issue order, how many waited for; reads in flight
    wait_barrier = {}   # load number -> barriers passed when its wait was executed
    barriers = 0
    regs, acc = {}, {}

    def val(t):
        return int(t, 0) if re.match(r"^-?(0x)?[0-9a-f]+$", t) else s.get(t, 0)

    pc, n = 0, 0
    while pc < len(lines):
        n += 1
        check(n < 200000, "does not end")
        ln = lines[pc]
        pc += 1
        if ln.endswith(":"):
            continue
        op, _, rest = ln.partition(" ")
        a = [t.strip() for t in rest.split(",")]
        if op == "s_mov_b32":
            s[a[0]] = val(a[1])
        elif op == "s_add_u32":
            s[a[0]] = val(a[1]) + val(a[2])
        elif op in ("s_cmp_gt_u32", "s_cmp_lt_u32", "s_cmp_eq_u32"):
            x, y = val(a[0]), val(a[1])
            scc = {"gt": x > y, "lt": x < y, "eq": x == y}[op[6:8]]
        elif op == "s_cselect_b32":
            s[a[0]] = val(a[1]) if scc else val(a[2])
        elif op == "s_cbranch_scc1":
            pc = labels[a[0]] if scc else pc
        elif op == "s_branch":
            pc = labels[a[0]]
        elif op == "buffer_load_dwordx4":
            which = "x" if a[1] == G.XRS else "w"
            so, off = a[2].split()[0], int(re.search(r"offset:(\d+)", ln).group(1))
            rec = s["s66" if which == "x" else "s70"]
            step, k = divmod(s[so], G.ROW)
            check(k == 0)
            check(bool(rec) == (step < steps), "records", which, step)
            i = int(a[0][1:]) - (g.xv if which == "x" else g.wv)
            check(i % 4 * 1024 == off, "instruction offset against the lane offset's", i, off)
            for w in range(4):
                at = (s["m0"] + off) // 1024 + per_wave[which] * w
                check(0 <= at * 1024 < g.lds)
                if at in free_after:   # the old content's reads returned before a barrier
                    check(free_after[at] is not None and free_after[at] < barriers,
                          "refilled while read", which, step, at)
                piece[at] = (which, step if rec else None, per_wave[which] * w + i, len(vm))
                free_after[at] = None if rec else -1
            vm.append((which, step))
        elif op == "ds_read_b128":
            reg, (v, off) = _span(a[0]), a[1].split()
            v, off = int(v[1:]), int(off.split(":")[1])
            which = "w" if v < g.rb else "x"
            base, u = divmod(v - (g.ra if which == "w" else g.rb), 2)
            blocks = g.na if which == "w" else g.mb
            got = set()
            for half in range(2):      # the waves of either half of the tile
                first = (off + 65536 * base) // 1024 + 2 * blocks * half
                for at in (first, first + 1):
                    check(at in piece, "read of an empty piece", ln)
                    kind, step, idx, num = piece[at]
                    check(kind == which and num in wait_barrier and wait_barrier[num] < barriers,
                          "read before its barrier", ln, step)
                    got.add((step, (idx // 2) - blocks * half))
            check(len(got) == 1, "rows of different steps", ln, got)
            step, blk = got.pop()
            lgkm.append((reg, (which, step, u, blk),
                         [(off + 65536 * base) // 1024 + 2 * blocks * h + e
                          for h in range(2) for e in range(2)]))
            for r in reg:
                regs[r] = "in flight"
        elif op == "s_waitcnt":
            m = re.search(r"vmcnt\((\d+)\)", ln)
            if m:
                while landed < len(vm) - int(m.group(1)):
                    wait_barrier[landed] = barriers
                    landed += 1
            m = re.search(r"lgkmcnt\((\d+)\)", ln)
            if m:
                while len(lgkm) > int(m.group(1)):
                    reg, what, ats = lgkm.pop(0)
                    for r in reg:
                        regs[r] = what
                    for at in ats:
                        free_after[at] = barriers
        elif op == "s_barrier":
            barriers += 1
        elif op == "v_mfma_f32_16x16x32_bf16":
            c, ra, rb = _span(a[0]), _span(a[1]), _span(a[2])
            check(a[3] == a[0])
            A, B = {regs.get(r) for r in ra}, {regs.get(r) for r in rb}
            check(len(A) == 1 and len(B) == 1 and not (A | B) & {None, "in flight"}, "operand", ln)
            (kw, sa, ua, na), (kx, sb, ub, mb) = A.pop(), B.pop()
            check((kw, kx) == ("w", "x") and sa == sb and ua == ub, "operands of two steps", ln)
            check(c[0] == 4 * (g.mb * na + mb), "accumulator of another block", ln)
            acc.setdefault(c[0], []).append((sa, ua))
        else:
            check(op in ("s_nop", "v_accvgpr_write_b32"), "unknown", ln)
    check(landed == len(vm) and not lgkm, "left in flight at the end")
    check(sorted(acc) == list(range(0, 4 * g.na * g.mb, 4)))
    for c, seq in acc.items():
        check(seq == [(t, u) for t in range(steps) for u in range(2)], "sum", c, seq)


def _lines(name):
    g = G.Gen(name)
    return g, [ln.replace("%=", "") for ln in g.generate()]


def test_generated_file_is_current():
    assert open(G.OUT).read() == G.render()


@pytest.mark.parametrize("name", list(G.VARIANTS))
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 6, 7, 11, 12, 13, 25])
def test_every_step_once_and_nothing_early(name, steps):
    g, lines = _lines(name)
    assert g.lds <= 163840 and g.n_vgpr <= 256
    replay(g, lines, steps)


def _drop(lines, match, skip=0):
    i = [k for k, ln in enumerate(lines) if re.match(match, ln)][skip]
    return lines[:i] + lines[i + 1:]


PLANTED = {
    "a wait one load short": lambda ls: [
        re.sub(r"vmcnt\((\d+)\) lgkmcnt", lambda m: f"vmcnt({int(m.group(1)) + 1}) lgkmcnt", ln)
        for ln in ls],
    "a barrier missing": lambda ls: _drop(ls, "s_barrier", 2),
    "an operand read missing": lambda ls: _drop(ls, "ds_read_b128", 30),
    "reads not waited for": lambda ls: _drop(ls, r"s_waitcnt lgkmcnt\(0\)", 1),
    "records kept past the end": lambda ls: [ln for ln in ls if ln != "s_cselect_b32 s66, s66, 0"],
    "a scalar offset not advanced": lambda ls: _drop(ls, f"s_add_u32 {G.SWO}", 1),
    "a slot one off": lambda ls: [ln.replace("%[m0x], ", "%[m0x], 1") if "%[m0x]" in ln else ln
                                  for ln in ls],
}


@pytest.mark.parametrize("name", list(G.VARIANTS))
@pytest.mark.parametrize("mistake", list(PLANTED))
def test_replay_finds_a_planted_mistake(name, mistake):
    g, lines = _lines(name)
    with pytest.raises(Wrong):
        replay(g, PLANTED[mistake](lines), 13)
