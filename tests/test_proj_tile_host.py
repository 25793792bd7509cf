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
TILES = ["8wave", "256x256", "256x224", "256x192", "256x160", "256x128", "128x128", "128x64"]

# (tile, tokens, channels, reduction, with norm and RoPE)
CASES = [
    ("256x256", 31885, 5120, 5120, 0), ("256x256", 32000, 15360, 5120, 1),
    ("256x128", 917, 5120, 5120, 0), ("256x192", 1152, 21504, 5376, 1),
    ("256x192", 4096, 5120, 5120, 0), ("8wave", 4096, 5120, 512, 0),
    ("256x192", 2048, 5120, 5120, 0), ("8wave", 2048, 5120, 960, 0),
    ("128x64", 300, 5120, 5120, 0), ("128x64", 1, 256, 64, 0),
    ("256x192", 768, 15360, 1536, 1), ("8wave", 768, 15360, 1472, 1),
    # test_gpu_proj_tiles.py
    ("256x256", 1000, 15360, 1088, 0), ("256x224", 801, 15360, 1024, 0),
    ("256x192", 700, 15360, 1152, 0), ("256x160", 600, 15360, 192, 0),
    ("256x128", 1001, 5120, 192, 0), ("256x128", 1001, 5120, 64, 0),
    ("256x128", 897, 5376, 320, 0), ("128x128", 400, 5120, 448, 0),
    ("128x64", 129, 256, 64, 0),
    ("256x256", 1024, 15360, 1536, 1), ("256x224", 1280, 21504, 1600, 1),
    ("256x192", 1024, 21504, 1536, 1), ("256x160", 1152, 15360, 1536, 1),
    ("256x160", 640, 15360, 128, 1), ("256x128", 1280, 5376, 256, 1),
    ("128x128", 1024, 2304, 704, 1), ("128x64", 256, 768, 64, 1),
]

HARNESS = r"""
#include "proj_tile.h"
#include <cstdio>
#include <cstdlib>
int main(int argc, char** argv) {
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
    subprocess.run([gxx, "-O1", "-std=c++17", f"-I{CSRC}", str(d / "t.cpp"), "-o", str(d / "t")],
                   check=True)

    def run(cases):
        args = [str(int(v)) for c in cases for v in c]
        out = subprocess.run([str(d / "t")] + args, check=True, capture_output=True, text=True)
        return [TILES[int(v)] for v in out.stdout.split()]
    return run


def test_named_sizes(pick):
    got = pick([c[1:] for c in CASES])
    assert got == [c[0] for c in CASES], [(c, g) for c, g in zip(CASES, got) if c[0] != g]


def test_few_steps_take_small_tiles_only_for_one_round(pick):
    cases = [(t, n, h, f) for t in (1, 130, 700, 2000, 9000) for n in (256, 1536, 5120, 15360)
             for h in (64, 512, 960) for f in (0, 1)]
    for (t, n, h, f), tile in zip(cases, pick(cases)):
        if tile != "8wave":
            tn, tm = map(int, tile.split("x"))
            assert tm <= 160
            assert -(-t // tm) * (n // tn) <= 256, (t, n, h, f, tile)
