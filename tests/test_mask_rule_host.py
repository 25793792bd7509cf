"""The lattice rules on tile pairs (csrc/mask_rule.h, compiled here with g++)
give the bitmap of their token-pair definition (the oracle's brute force):
LOCAL and AXIAL over one-token rows and frames, ragged ends, prefixes that end
inside and at the edge of a tile, wide windows, spatial tiles larger than the
frame, landmarks, and drawn lattices."""
import ctypes
import os
import random
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "minimax-h3-swift_amd", "csrc")

HARNESS = r"""
#include "mask_rule.h"
using namespace h3hip;
// Calls of the header's functions (g++ -finstrument-functions).
static long calls = 0;
extern "C" {
__attribute__((no_instrument_function)) void __cyg_profile_func_enter(void*, void*) { calls++; }
__attribute__((no_instrument_function)) void __cyg_profile_func_exit(void*, void*) {}
__attribute__((no_instrument_function)) long take_calls() {
  const long c = calls;
  calls = 0;
  return c;
}
}
extern "C" void bitmap(const int32_t* p, const uint8_t* landmark, uint8_t* out) {
  const RuleDev r{p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], p[9], 0, p[10], nullptr,
                  landmark};
  for (int32_t q = 0; q < r.n_tiles; q++) {
    RuleBox box[kMaxBoxes] = {};
    const TileSpan s = tile_span(r, q);
    if (r.kind == H3HIP_RULE_LOCAL && !tile_in_prefix(r, q)) tile_boxes(r, s, box);
    for (int32_t k = 0; k < r.n_tiles; k++)
      out[q * r.n_tiles + k] = tile_in_prefix(r, q) || tile_in_prefix(r, k) ||
                               lattice_tiles_see(r, s, tile_span(r, k), box);
  }
}
"""

LOCAL, AXIAL = 2, 3
# (kind, prefix, frames, height, width, frame window, spatial tile, spatial window, landmarks)
CASES = [
    (LOCAL, 637, 5, 24, 42, 1, (8, 8), 1, ()),
    (LOCAL, 0, 700, 1, 1, 3, (8, 8), 0, (5,)),        # one token a frame
    (LOCAL, 128, 3, 300, 1, 0, (7, 1), 2, ()),        # one token a row, prefix of one tile
    (LOCAL, 127, 2, 1, 500, 0, (1, 3), 5, ()),        # one row a frame
    (LOCAL, 129, 9, 13, 22, 100, (50, 60), 0, ()),    # windows over everything
    (LOCAL, 1, 1, 40, 40, 0, (1, 1), 0, ()),          # only the token itself
    (LOCAL, 300, 11, 9, 16, 0, (8, 8), 0, (0, 10)),
    (AXIAL, 746, 9, 15, 27, 1, (8, 8), 1, (0, 4, 8)),
    (AXIAL, 0, 900, 1, 1, 1, (8, 8), 1, ()),
    (AXIAL, 5, 3, 1, 127, 1, (8, 8), 1, ()),          # frames one token short of a tile
    (AXIAL, 0, 4, 16, 16, 1, (8, 8), 1, ()),          # frames of whole tiles
    (AXIAL, 200, 2, 1, 1, 1, (8, 8), 1, (1,)),
]


def _drawn(n):
    rng = random.Random(17)
    out = []
    while len(out) < n:
        f, h, w = rng.randint(1, 40), rng.randint(1, 30), rng.randint(1, 45)
        if f * h * w > 3000:
            continue
        lm = tuple(sorted(rng.sample(range(f), rng.randint(0, min(2, f)))))
        out.append((rng.choice([LOCAL, AXIAL]), rng.randint(0, 400), f, h, w, rng.randint(0, 2),
                    (rng.randint(1, 9), rng.randint(1, 9)), rng.randint(0, 2), lm))
    return out


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("mask_rule")
    src, so = d / "h.cpp", d / "h.so"
    src.write_text(HARNESS)
    subprocess.run([cxx, "-O1", "-std=c++17", "-fPIC", "-shared", "-finstrument-functions",
                    "-Wl,-Bsymbolic", "-I", CSRC, str(src), "-o",
                    str(so)], check=True)
    lib = ctypes.CDLL(str(so))
    lib.take_calls.restype = ctypes.c_long
    return lib


def _bitmap(rules, rule, f, sp, fw, sw, lm):
    flags = np.zeros(f, np.uint8)
    flags[list(lm)] = 1
    p = np.array([rule.kind, rule.seq_len, rule.prefix_len, f, rule.height, rule.width, fw, sp[0],
                  sp[1], sw, rule.n_tiles], np.int32)
    got = np.zeros((rule.n_tiles, rule.n_tiles), np.uint8)
    u8 = ctypes.POINTER(ctypes.c_uint8)
    rules.bitmap(p.ctypes.data_as(ctypes.POINTER(ctypes.c_int32)),
                 flags.ctypes.data_as(u8) if lm else None, got.ctypes.data_as(u8))
    return got


@pytest.mark.parametrize("case", CASES + _drawn(40))
def test_tile_pairs_match_token_pairs(rules, orc, case):
    kind, prefix, f, h, w, fw, sp, sw, lm = case
    seq = prefix + f * h * w
    rule = orc.Rule(kind, seq, prefix_len=prefix, frames=f, height=h, width=w, frame_window=fw,
                    sp_tile=sp, sp_window=sw, landmarks=list(lm))
    got = _bitmap(rules, rule, f, sp, fw, sw, lm)
    assert np.array_equal(got, orc.tile_bitmap(rule))


@pytest.mark.parametrize("f,h,w", [(2048, 1, 1), (1, 2048, 1), (16, 128, 1), (256, 2, 4),
                                   (128, 4, 4), (32, 8, 8), (2, 32, 32)])
def test_a_tile_pair_costs_the_same_however_narrow_the_lattice(rules, orc, f, h, w):
    """LOCAL with windows that see only the token itself, so that nothing ends
    the comparison early: 5 x 5 boxes of three axes each. (Row by row, a
    pair of tiles of one-token rows is 16,384 comparisons.)"""
    rule = orc.Rule(LOCAL, f * h * w, frames=f, height=h, width=w, frame_window=0,
                    sp_tile=(1, 1), sp_window=0)
    rules.take_calls()
    got = _bitmap(rules, rule, f, (1, 1), 0, 0, ())
    calls = rules.take_calls()
    assert np.array_equal(got, orc.tile_bitmap(rule))
    assert 0 < calls <= (25 * 5 + 64) * got.size, calls / got.size
