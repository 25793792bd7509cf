"""Plans of half units (64 queries, bsattn_half_kernel) against the oracle: plans of
one half unit per workgroup up to the last that still fits, several on a
workgroup with empty rows between them, a few long rows among short ones, and
sequences that end in either half of the last tile; and the same heads on plans of
whole units, bit for bit. Every row of every head up to 3,000 tokens, of three
heads beyond.

Bars of the attention tests: max-abs 2e-2, mean-abs 2e-3 against fp32."""
import numpy as np
import pytest

from _gpu import bits, err_stats, f32, head_major_inputs, note

pytestmark = pytest.mark.gpu


def _bitmap(kind, n, rng):
    if kind == "dense":
        return np.ones((n, n), np.uint8)
    bm = (rng.random((n, n)) < 0.25).astype(np.uint8)
    if kind in ("long", "gaps"):   # one full row among rows of one tile
        bm[:] = 0
        bm[np.arange(n), np.arange(n)] = 1
        bm[0] = 1
        if kind == "gaps":         # two rows of three without a tile
            bm[np.arange(n) % 3 > 0] = 0
    else:
        bm[n // 2] = 0          # a row with no active tile
    return bm


# (tokens, heads, rows, queries of a unit)
CASES = [
    (1, 1, "dense", 64), (63, 2, "dense", 64), (64, 1, "dense", 64), (65, 3, "dense", 64),
    (128, 1, "dense", 64), (193, 2, "sparse", 64),
    (917, 16, "dense", 64),      # 128 units: one half unit on each of 256 CUs
    (1000, 17, "sparse", 128),   # 136: two half units on some would end later
    (2500, 3, "sparse", 64), (4000, 4, "long", 64),
    (8000, 6, "long", 64),       # 756 half units: three on most workgroups
    (8000, 6, "gaps", 64),       # the same with empty rows between
]


@pytest.mark.parametrize("S,heads,kind,unit_rows", CASES)
def test_every_row(h3, orc, S, heads, kind, unit_rows):
    from h3hip import _lib as L, ops
    note(f"half units S={S} heads={heads} {kind}")
    n = (S + 127) // 128
    bm = _bitmap(kind, n, np.random.default_rng(S))
    plan = h3.TilePlan(h3.MaskRule.from_bitmap(S, bm), heads=heads)
    assert plan.schedule()[0] == unit_rows
    q, k, v = head_major_inputs(heads, S, n * 128, 128, S, pad_value=float("nan"))
    out = ops.bsattn_fwd(plan, q, k, v)
    tok = ops.bsattn_fwd(plan, q, k, v, out_layout=L.OUT_TOKEN_MAJOR)
    assert np.array_equal(bits(out), bits(tok.view(-1, heads, 128).transpose(0, 1)))
    got = f32(out)
    assert np.all(got[:, S:] == 0)
    for i in np.flatnonzero(bm.sum(1) == 0):
        assert np.all(got[:, i * 128:(i + 1) * 128] == 0), i
    hs = range(heads) if S < 3000 else (0, heads // 2, heads - 1)
    for h in hs:
        want = orc.attend_masked(f32(q)[h:h + 1, :S], f32(k)[h:h + 1, :S], f32(v)[h:h + 1, :S],
                                 128 ** -0.5, bm)
        mx, mean = err_stats(got[h:h + 1, :S], want)
        assert mx <= 2e-2 and mean <= 2e-3, (h, mx, mean)


# (tokens, heads, heads of a plan of whole units, rows)
PAIRS = [(100, 4, 200, "dense"), (917, 8, 24, "dense"), (1000, 5, 40, "sparse"),
         (8000, 6, 30, "gaps")]


@pytest.mark.parametrize("S,heads,more,kind", PAIRS)
def test_bits_of_whole_units(h3, S, heads, more, kind):
    """The first `heads` heads of a plan of `more`, which runs whole units."""
    from h3hip import ops
    note(f"half against whole units S={S} heads={heads}, {more} {kind}")
    n = (S + 127) // 128
    rule = h3.MaskRule.from_bitmap(S, _bitmap(kind, n, np.random.default_rng(S)))
    half, whole = h3.TilePlan(rule, heads=heads), h3.TilePlan(rule, heads=more)
    assert half.schedule()[0] == 64 and whole.schedule()[0] == 128
    q, k, v = head_major_inputs(more, S, n * 128, 128, S)
    want = ops.bsattn_fwd(whole, q, k, v)
    got = ops.bsattn_fwd(half, *(t[:heads].contiguous() for t in (q, k, v)))
    assert np.array_equal(bits(got), bits(want[:heads]))
