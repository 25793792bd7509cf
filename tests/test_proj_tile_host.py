"""The rule that picks a projection's kernel and tile (csrc/proj_tile.h, compiled
here with g++): every size gets a tile that divides its channels, the larger
tile where it needs no more time in rounds, the eight-wave kernel for short
reductions, and the sizes test_gpu_proj_tiles.py runs get the tile they name."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "minimax-h3-swift_amd", "csrc")
TILES = ["8wave", "256x256", "256x224", "256x192", "256x160", "256x128", "128x192", "128x160",
         "128x128", "128x64"]

# (tile, tokens, channels, reduction, with norm and RoPE)
CASES = [
    ("256x256", 31885, 5120, 5120, 0), ("256x256", 32000, 15360, 5120, 1),
    ("128x160", 917, 5120, 5120, 0), ("256x192", 1152, 21504, 5376, 1),
    ("256x192", 4096, 5120, 5120, 0), ("8wave", 4096, 5120, 512, 0),
    ("256x192", 2048, 5120, 5120, 0), ("8wave", 2048, 5120, 960, 0),
    ("128x64", 300, 5120, 5120, 0), ("128x64", 1, 256, 64, 0),
    ("256x192", 768, 15360, 1536, 1), ("8wave", 768, 15360, 1472, 1),
    # test_gpu_proj_tiles.py
    ("256x256", 1000, 15360, 1088, 0), ("256x224", 801, 15360, 1024, 0),
    ("256x192", 700, 15360, 1152, 0), ("256x160", 600, 15360, 192, 0),
    ("256x128", 1201, 5120, 192, 0), ("256x128", 1201, 5120, 64, 0),
    ("256x128", 1160, 5376, 320, 0), ("128x192", 1001, 5120, 192, 0),
    ("128x160", 900, 5120, 320, 0), ("128x128", 400, 5120, 448, 0),
    ("128x64", 129, 256, 64, 0),
    ("256x256", 1024, 15360, 1536, 1), ("256x224", 1280, 21504, 1600, 1),
    ("256x192", 1024, 21504, 1536, 1), ("256x160", 1152, 15360, 1536, 1),
    ("256x160", 640, 15360, 128, 1), ("256x128", 1280, 5376, 256, 1),
    ("128x192", 384, 15360, 704, 1), ("128x160", 896, 5376, 256, 1),
    ("128x128", 1024, 2304, 704, 1), ("128x64", 256, 768, 64, 1),
]

HARNESS = r"""
#include "proj_tile.h"
#include <cstdio>
#include <cstdlib>
#include <set>
// Calls of the headers' functions (g++ -finstrument-functions).
static long calls = 0;
extern "C" {
__attribute__((no_instrument_function)) void __cyg_profile_func_enter(void*, void*) { calls++; }
__attribute__((no_instrument_function)) void __cyg_profile_func_exit(void*, void*) {}
}
int main(int argc, char** argv) {
  if (argc > 1 && argv[1][0] == 'g') {   // grids: every tile once, longest list as stated
    for (int a = 2; a + 3 < argc; a += 4) {
      const h3hip::ProjGrid g = h3hip::proj_grid(std::atoi(argv[a]), std::atoi(argv[a + 1]),
                                                 std::atoi(argv[a + 2]), std::atoi(argv[a + 3]));
      std::set<long> seen;
      int n = 0, longest = 0;
      for (int x = 0; x < h3hip::kOrderXcds; x++) {
        longest = std::max(longest, g.order.length(x));
        for (int p = 0; p < g.order.length(x); p++, n++) {
          const auto t = g.order.tile(x, p);
          const int tm = (int)(t >> 16), tn = (int)(t & 0xffff);   // as the kernels read it
          if (tm >= 0 && tm < g.order.tiles_m && tn < g.order.tiles_n) seen.insert(t);
        }
      }
      std::printf("%d %d %d\n", n == g.order.tiles_m * g.order.tiles_n && n == (int)seen.size() &&
                  longest == g.longest, g.order.chunk, g.rounds);
    }
    return 0;
  }
  if (argc > 1 && argv[1][0] == 'c') {   // function calls of a pick
    for (int a = 2; a + 3 < argc; a += 4) {
      const int v[4] = {std::atoi(argv[a]), std::atoi(argv[a + 1]), std::atoi(argv[a + 2]),
                        std::atoi(argv[a + 3])};
      calls = 0;
      h3hip::pick_proj_tile(v[0], v[1], v[2], v[3] != 0);
      std::printf("%ld\n", calls);
    }
    return 0;
  }
  for (int a = 1; a + 3 < argc; a += 4)
    std::printf("%d\n", (int)h3hip::pick_proj_tile(std::atoi(argv[a]), std::atoi(argv[a + 1]),
                                                   std::atoi(argv[a + 2]), std::atoi(argv[a + 3]) != 0));
}
"""


@pytest.fixture(scope="module")
def pick(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not found")
    d = tmp_path_factory.mktemp("tile")
    (d / "t.cpp").write_text(HARNESS)
    subprocess.run([gxx, "-O1", "-std=c++17", "-finstrument-functions", f"-I{CSRC}",
                    str(d / "t.cpp"), "-o", str(d / "t")], check=True)

    def run(cases):
        args = [str(int(v)) for c in cases for v in c]
        out = subprocess.run([str(d / "t")] + args, check=True, capture_output=True, text=True)
        return [TILES[int(v)] for v in out.stdout.split()]

    def grids(cases):
        args = [str(int(v)) for c in cases for v in c]
        out = subprocess.run([str(d / "t"), "g"] + args, check=True, capture_output=True, text=True)
        return [tuple(map(int, ln.split())) for ln in out.stdout.splitlines()]

    def costs(cases):
        args = [str(int(v)) for c in cases for v in c]
        out = subprocess.run([str(d / "t"), "c"] + args, check=True, capture_output=True, text=True)
        return [int(v) for v in out.stdout.split()]
    run.grids, run.costs = grids, costs
    return run


def test_named_sizes(pick):
    got = pick([c[1:] for c in CASES])
    assert got == [c[0] for c in CASES], [(c, g) for c, g in zip(CASES, got) if c[0] != g]


def test_sizes_of_the_eight_wave_tests(pick):
    """What test_gpu_proj_eight_waves.py runs picks that kernel, and the row subsets
    it compares with do not."""
    import test_gpu_proj_eight_waves as t
    whole = [(-(-S // 128) * 128, 384 * H, k, f) for S, k, H, *_ in t.QKV for f in (0, 1)]
    whole += [(S, n, k, 0) for S, k, n, *_ in t.OUT]
    parts = [(128, 384 * H, k, 0) for _, k, H, *_ in t.QKV] + [(t.ROWS, n, k, 0)
                                                                for _, k, n, *_ in t.OUT]
    assert pick(whole) == ["8wave"] * len(whole)
    assert "8wave" not in pick(parts), pick(parts)


def test_few_steps_take_small_tiles_only_for_one_round(pick):
    cases = [(t, n, h, f) for t in (1, 130, 700, 2000, 9000) for n in (256, 1536, 5120, 15360)
             for h in (64, 512, 960) for f in (0, 1)]
    for (t, n, h, f), tile in zip(cases, pick(cases)):
        if tile != "8wave":
            tn, tm = map(int, tile.split("x"))
            assert tm <= 160
            assert -(-t // tm) * (n // tn) <= 256, (t, n, h, f, tile)


def test_launch_orders_list_every_tile_once(pick):
    """(tokens, channels, tile tokens, tile channels): the chunk that needs the
    fewest rounds, 252 tiles in one; every tile once in each order."""
    cases = [(896, 5376, 160, 128), (31885, 15360, 256, 256), (1, 256, 64, 128),
             (1152, 21504, 192, 256), (917, 5120, 160, 128), (300, 5120, 64, 128),
             (641, 15360, 160, 256), (2048, 5120, 192, 256), (18102, 5376, 224, 256),
             (8388609, 256, 256, 256), (16776960, 256, 256, 256), (256, 16776960, 256, 256)]
    got = pick.grids(cases)
    assert all(ok for ok, _, _ in got), got
    assert got[0][2] == 1 and got[0][1] < 4
    assert got[1][1] == 4                      # many rounds: the chunk that shares the most
    for (t, n, tt, tn), (_, chunk, rounds) in zip(cases, got):
        tiles = -(-t // tt) * (n // tn)
        assert rounds <= -(-tiles // 256) + (tiles > 256 * 0.95), (t, n, chunk, rounds)


def test_picking_is_cheap(pick):
    """Every projection call picks a tile: nine shapes, one launch order each and
    up to two more, two lists of an order counted. (All lists of three orders
    are 1,522 calls and 0.9 us, of a call of 8 us.)"""
    costs = pick.costs([c[1:] for c in CASES])
    assert 0 < min(costs) and max(costs) <= 9 * 3 * 20, costs
    assert sorted(costs)[len(costs) // 2] <= 9 * 1.5 * 20, costs
