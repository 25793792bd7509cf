"""Plans of half units (64 queries, bsattn_half_kernel) against the oracle, every
row of every head: plans of one half unit per workgroup up to the last that
still fits, the first that does not, a few long rows among short ones, empty
rows, and sequences that end in either half of the last tile.

Bars of the attention tests: max-abs 2e-2, mean-abs 2e-3 against fp32."""
import numpy as np
import pytest

from _gpu import bits, err_stats, f32, head_major_inputs, note

pytestmark = pytest.mark.gpu


def _bitmap(kind, n, rng):
    if kind == "dense":
        return np.ones((n, n), np.uint8)
    bm = (rng.random((n, n)) < 0.25).astype(np.uint8)
    if kind == "long":          # one full row among rows of a tile or two
        bm[:] = 0
        bm[np.arange(n), np.arange(n)] = 1
        bm[0] = 1
    else:
        bm[n // 2] = 0          # a row with no active tile
    return bm


@pytest.mark.parametrize("S,heads,kind", [
    (1, 1, "dense"), (63, 2, "dense"), (64, 1, "dense"), (65, 3, "dense"), (128, 1, "dense"),
    (193, 2, "sparse"), (917, 16, "dense"),    # 128 units: one half unit on each of 256 CUs
    (1000, 17, "sparse"),                      # 136: two half units on some
    (2500, 3, "sparse"), (4000, 4, "long"), (8000, 6, "long"),
])
def test_every_row(h3, orc, S, heads, kind):
    from h3hip import _lib as L, ops
    note(f"half units S={S} heads={heads} {kind}")
    n = (S + 127) // 128
    bm = _bitmap(kind, n, np.random.default_rng(S))
    plan = h3.TilePlan(h3.MaskRule.from_bitmap(S, bm), heads=heads)
    q, k, v = head_major_inputs(heads, S, n * 128, 128, S, pad_value=float("nan"))
    out = ops.bsattn_fwd(plan, q, k, v)
    tok = ops.bsattn_fwd(plan, q, k, v, out_layout=L.OUT_TOKEN_MAJOR)
    assert np.array_equal(bits(out), bits(tok.view(-1, heads, 128).transpose(0, 1)))
    got = f32(out)
    assert np.all(got[:, S:] == 0)
    hs = range(heads) if S < 3000 else (0, heads - 1)
    for h in hs:
        want = orc.attend_masked(f32(q)[h:h + 1, :S], f32(k)[h:h + 1, :S], f32(v)[h:h + 1, :S],
                                 128 ** -0.5, bm)
        mx, mean = err_stats(got[h:h + 1, :S], want)
        assert mx <= 2e-2 and mean <= 2e-3, (h, mx, mean)
