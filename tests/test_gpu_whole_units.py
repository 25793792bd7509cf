"""The edge and drawn cases of test_gpu_attention_edges.py and
test_gpu_attention_random.py on plans of whole units (128 queries,
bsattn_fwd_kernel, which serves every large plan). With their few heads those
plans run half units; with more than six units a workgroup a plan runs whole ones,
so here each case has 1,537 units or more, six or seven one after another on each
workgroup. Three heads of each are compared with the oracle, all rows, at the same
bars (max-abs 2e-2, mean-abs 2e-3)."""
import math

import numpy as np
import pytest
import torch

from _gpu import err_stats, f32, head_major_inputs, note, randn_bf16_gpu
from test_gpu_attention_random import _case

pytestmark = pytest.mark.gpu

MAX_ABS, MEAN_ABS = 2e-2, 2e-3
UNITS = 6 * 256 + 1


def _check(h3, orc, S, bm, q, k, v, scale, layout=0):
    from h3hip import ops
    n, heads = len(bm), q.shape[0]
    plan = h3.TilePlan(h3.MaskRule.from_bitmap(S, bm), heads=heads)
    assert plan.schedule()[0] == 128
    out = ops.bsattn_fwd(plan, q, k, v, scale, out_layout=layout)
    torch.cuda.synchronize()
    if layout == 1:
        out = out.view(n * 128, heads, 128).transpose(0, 1)
    else:
        assert torch.all(out[:, S:] == 0)
    assert torch.isfinite(out[:, :S].float()).all()
    for i in np.flatnonzero(bm.sum(1) == 0):
        assert torch.all(out[:, i * 128:min((i + 1) * 128, S)] == 0), i
    hs = [0, heads // 2, heads - 1]
    want = orc.attend_masked(*(f32(t[hs])[:, :S] for t in (q, k, v)), scale, bm, tile=128)
    mx, mean = err_stats(f32(out[hs])[:, :S], want)
    print(f"max-abs {mx:.2e} mean-abs {mean:.2e}")
    assert mx < MAX_ABS and mean < MEAN_ABS, (mx, mean)


def _heads(n):
    return -(-UNITS // n)


@pytest.mark.parametrize("scale", [0.088, 1.0])
@pytest.mark.parametrize("S", [1, 5, 64, 127, 128, 129, 192, 256, 257, 300])
def test_short_and_boundary_lengths(h3, orc, S, scale):
    """Among them lengths whose last tile has at most 64 valid keys, so that one
    64-key half sees padding only."""
    n = (S + 127) // 128
    note(f"whole units S={S} H={_heads(n)} scale={scale}")
    q, k, v = head_major_inputs(_heads(n), S, n * 128, 128, S + 3, pad_value=float("nan"))
    _check(h3, orc, S, np.ones((n, n), np.uint8), q, k, v, scale)


@pytest.mark.parametrize("q_scale,ramp", [(6.0, 0.0), (1.0, 6.0), (4.0, 4.0)])
def test_rising_maxima_force_rescales(h3, orc, q_scale, ramp):
    S, n = 900, 8
    note(f"whole units rising maxima q_scale={q_scale} ramp={ramp}")
    q, k, v = head_major_inputs(_heads(n), S, n * 128, 128, 17)
    q, k = ((t.float() * q_scale).to(torch.bfloat16) for t in (q, k))
    if ramp:   # every later tile holds a larger maximum
        up = torch.linspace(0, ramp, n * 128, device="cuda")[None, :, None]
        k = (k.float() + up * q.float().mean(dim=1, keepdim=True).sign()).to(torch.bfloat16)
    k[:, S:] = 0
    _check(h3, orc, S, np.ones((n, n), np.uint8), q, k, v, 1.0 / math.sqrt(128))


@pytest.mark.parametrize("scale", [0.088, 0.125, 1.0])
def test_row_whose_only_tile_is_the_ragged_last(h3, orc, scale):
    n = 5
    S = (n - 1) * 128 + 40
    bm = np.eye(n, dtype=np.uint8)
    bm[0] = 1
    bm[2] = bm[n - 1]
    note(f"whole units, rows of the ragged last tile only, scale={scale}")
    _check(h3, orc, S, bm, *head_major_inputs(_heads(n), S, n * 128, 128, 41), scale)


@pytest.mark.parametrize("seed", range(16))
def test_drawn_case(h3, orc, seed):
    n, S, _, bm, scale, magnitude, pad, layout = _case(seed)
    note(f"whole units seed={seed} n={n} S={S} H={_heads(n)} density={bm.mean():.2f} "
         f"scale={scale:.3f} magnitude={magnitude} pad={pad} layout={layout}")
    shape = (_heads(n), n * 128, 128)
    q, k = (randn_bf16_gpu(shape, 50 * seed + i, magnitude) for i in range(2))
    v = randn_bf16_gpu(shape, 50 * seed + 2)
    for t in (q, k, v):
        t[:, S:] = pad
    _check(h3, orc, S, bm, q, k, v, scale, layout)
