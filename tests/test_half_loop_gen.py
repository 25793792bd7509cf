"""The tile loop of half units (csrc/gen_half_loop.py -> csrc/bsattn_half_loop.inc):
it is current, stays within its registers, and passes the hazard scans of
test_tile_loop_gen.py, which are tested there; and it loads each of a tile's 128
rows once, into the place the operand reads expect it."""
import importlib.util
import os
import re

import pytest

import test_tile_loop_gen as T

CSRC = T.CSRC


@pytest.fixture(scope="module")
def gen():
    spec = importlib.util.spec_from_file_location("gen_half_loop",
                                                  os.path.join(CSRC, "gen_half_loop.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m.load()


@pytest.fixture(scope="module")
def lines(gen):
    return gen.generate()


def test_include_is_current(gen):
    assert open(gen.OUT).read() == gen.render(), "run python3 gen_half_loop.py in csrc/"


def test_registers_do_not_overlap(gen, lines):
    offsets = list(range(gen.KA0, gen.KA0 + 8)) + list(range(gen.VA0, gen.VA0 + 8))
    offsets += list(range(gen.DK0, gen.DK0 + gen.LOADS)) + list(range(gen.DV0, gen.DV0 + gen.LOADS))
    temps = [gen.MX, gen.SW, gen.AL, gen.LA, gen.LB]
    assert len(set(offsets + temps + [gen.M, gen.L])) == len(offsets) + len(temps) + 2
    assert max(offsets + temps) < gen.N_VGPR <= 256
    written = {r for ln in lines if ln.startswith("v_") and not ln.startswith(("v_mfma", "v_cmp"))
               for r in T._regs(T._split(ln)[1][0])}
    assert not written & {("v", r) for r in offsets}


def test_hazard_scans(gen, lines):
    assert T.exp_read_next(lines) == []
    assert T.permlane_unsettled(lines) == []
    assert T.m0_unsettled(lines) == []
    assert T.ring_overwritten(gen, lines) == []
    assert T.mfma_read_soon(lines) == []
    assert T.ring_unwaited(gen, lines) == []


@pytest.mark.parametrize("which", ["k", "v"])
@pytest.mark.parametrize("slot", [0, 1])
def test_loads_cover_the_wave_rows_once(gen, which, slot):
    """Load i of wave w moves rows 32w + 4i .. +3 to 256 (32w + 4i) of the slot:
    M0 and the instruction offset give the LDS address, and the lane offset,
    lowered by 1024 (i & 3), gives the row."""
    m0 = None
    seen = []
    for group in gen.dma_lines(which, slot):
        for ln in group:
            m = re.match(r"s_add_u32 m0, %\[m0[kv]\], (\d+)", ln)
            if m:
                m0 = int(m.group(1))
            m = re.match(r"buffer_load_dwordx4 v(\d+), .* offset:(\d+) lds", ln)
            if m:
                i, off = int(m.group(1)) - (gen.DK0 if which == "k" else gen.DV0), int(m.group(2))
                assert off == 1024 * (i & 3) < 4096
                assert m0 + off == slot * gen.KSLOT + 256 * 4 * i
                seen.append(i)
    assert seen == list(range(8))
