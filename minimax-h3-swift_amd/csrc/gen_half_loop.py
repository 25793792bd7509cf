#!/usr/bin/env python3
"""Writes bsattn_half_loop.inc: the tile loop of bsattn_half_kernel, whose work
units are 64 queries. It is gen_tile_loop.py's stream on four waves instead of
eight: wave w owns queries 32(w & 1) .. +31 and key half w >> 1, and loads 32
rows of each K and V tile instead of 16. One wave per SIMD leaves twice the
registers, which hold the four more lane offsets of each tile's loads.

Registers that differ: v[114:121] and v[122:129] the K and V load offsets,
v[130:134] the softmax temporaries.

Run `python3 gen_half_loop.py` in this directory after editing either
generator; the generated file is committed, and tests/test_half_loop_gen.py
checks it is current.
"""
from __future__ import annotations

import importlib.util
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))


def load():
    """gen_tile_loop with this loop's layout (its functions read the layout
    from their module's globals)."""
    spec = importlib.util.spec_from_file_location("half_loop", os.path.join(HERE, "gen_tile_loop.py"))
    g = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(g)
    g.OUT = os.path.join(HERE, "bsattn_half_loop.inc")
    g.SOURCE, g.MACRO = "gen_half_loop.py", "H3_HALF_LOOP"
    g.WAVES, g.ROWS_PER_WAVE, g.LOADS = 4, 32, 8
    g.DV0 = g.DK0 + g.LOADS
    g.MX, g.SW, g.AL, g.LA, g.LB = range(g.DV0 + g.LOADS, g.DV0 + g.LOADS + 5)
    g.T4 = (g.MX, g.SW, g.AL, g.LB)
    g.N_VGPR = g.LB + 1
    return g


if __name__ == "__main__":
    sys.exit(load().main())
