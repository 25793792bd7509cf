"""The workloads this library is timed on, through its public entry points.

The library is one DiT attention layer's hot path: the mask -> tile-list
builder, the Q/K norm + RoPE prologue, block-sparse attention, and the two
projections around them. A program builds a ``TilePlan`` and a rotation table
once per shape, keeps its weights on the GPU, and then calls one entry point
per layer and sampling step. The sizes are this repository's configurations
(``h3hip.configs``: cfg1 to cfg4 and the reference's axial shape) and the same
packings with a single latent frame, which is what a still image or the first
frame of a clip is; ``draw`` spreads over the clips in between.

``exact`` restates each path in float64 with torch alone.
"""
from __future__ import annotations

import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("minimax-h3-swift_amd"))

import h3hip  # noqa: E402
from h3hip import _lib as L, ops  # noqa: E402
from h3hip.backend import AttentionContext, H3HIPBackend, sdpa  # noqa: E402
from h3hip.layer import AttentionLayer, RopeState  # noqa: E402

D = 128
T = 128                       # tokens per tile
EPS = 1e-6
DEV = "cuda:0"
PAIR_DIMS = {128: (32, 48, 48), 96: (32, 32, 32)}   # rot -> t, h, w channels


# ------------------------------------------------------------------ the cases

def _case(name, op, rule, prefix, frames, height, width, heads, **kw):
    c = dict(name=name, op=op, rule=rule, prefix=prefix, frames=frames, height=height,
             width=width, heads=heads)
    c.update(kw)
    return c


def listed():
    return [
        # A render starts: the tile lists and the schedule of the 1344x768, 5 s
        # shape are built, once per shape, with two keyframes every token sees.
        _case("plan_local_31885", "plan", "local", 637, 31, 24, 42, 40),
        # One frame of 864x480 behind its text: the smallest call a sampler
        # makes, the prologue at launch-latency size.
        _case("prologue_917x40", "prologue", "dense", 512, 1, 15, 27, 40, rot=128, fp32=False),
        # The prologue of the headline clip (Q and K of a fused qkv).
        _case("prologue_31885x40", "prologue", "local", 637, 31, 24, 42, 40, rot=128, fp32=False),
        # The plumbing-size layer: 4 heads, 4,096 tokens, a band of tiles.
        _case("attn_band_4096x4", "attention", "band", 0, 4, 32, 32, 4, entry="head_major"),
        # One frame, everything attends to everything, ragged last tile.
        _case("attn_dense_917x40", "attention", "dense", 512, 1, 15, 27, 40, entry="strided"),
        # The headline layer: local window, Q and K head-major from the
        # prologue, V read in place from the fused qkv.
        _case("attn_local_31885x40", "attention", "local", 637, 31, 24, 42, 40, entry="strided"),
        # The dense path at the 864x480, 7 s shape ("faithful" quality).
        _case("attn_dense_18102x40", "attention", "dense", 687, 43, 15, 27, 40,
              entry="head_major"),
        # The reference's axial topology at its production shape, through the
        # seam the reference's layer calls, on [S, H, D] arrays.
        _case("attn_axial_15731x56", "attention", "axial", 746, 37, 15, 27, 56, entry="sdpa"),
        # QKV with norm and RoPE for one frame at the reference model's width.
        _case("qkv_1151x5376", "qkv", "dense", 746, 1, 15, 27, 56, hidden=5376, rot=96,
              fp32=False),
        # QKV with norm and RoPE for the headline clip.
        _case("qkv_31885x5120", "qkv", "local", 637, 31, 24, 42, 40, hidden=5120, rot=128,
              fp32=False),
        # The out-projection for one frame.
        _case("out_proj_917x5120", "out_proj", "dense", 512, 1, 15, 27, 40, hidden=5120),
        # A whole attention layer of the 864x480, 7 s clip: projection with
        # norm and RoPE, local attention, out-projection.
        _case("layer_local_18102x40", "layer", "local", 687, 43, 15, 27, 40, hidden=5120,
              rot=128, fp32=False, projection="fused"),
    ]


# The dearest listed case of each kind: no drawn case costs more.
_CAP = {"plan": 250 * 250, "prologue": 31885 * 40, "attention": 20164 * 40,
        "qkv": 31885 * 5120 * 15360, "out_proj": 31885 * 5120 * 5120, "layer": 18102 * 5120 * 20480}


def draw(rng):
    """One more case: any of the paths, a clip between one small frame and the
    headline shape (token counts spread over their logarithm), either model
    width, the options a caller picks."""
    while True:
        op = rng.choice(["plan", "prologue", "prologue", "attention", "attention", "attention",
                         "qkv", "qkv", "out_proj", "out_proj", "layer"])
        height, width = rng.choice([(15, 27), (24, 42), (27, 15), (32, 32), (13, 22), (9, 16)])
        tokens = math.exp(rng.uniform(math.log(300), math.log(31885)))
        prefix = rng.choice([0, rng.randint(1, 900), 512 + rng.randint(0, 250)])
        frames = max(1, int((tokens - prefix) / (height * width)))
        h3 = rng.random() < 0.3
        c = dict(op=op, rule="dense", prefix=prefix, frames=frames, height=height, width=width,
                 heads=56 if h3 else 40)
        hidden, rot = (5376, 96) if h3 else (5120, 128)
        seq = prefix + frames * height * width
        if op in ("plan", "attention", "layer"):
            c["rule"] = rng.choice(["local", "local", "dense", "axial", "band"])
        if op == "plan" and (c["rule"] == "dense" or frames < 8 or _tiles(c) < 8):
            continue
        if op in ("plan", "prologue", "attention") and rng.random() < 0.3:
            c["heads"] = rng.choice([2, 4, 5, 8, 24])
        fp32 = rng.random() < 0.15
        if op == "plan":
            cost = _tiles(c) ** 2
        elif op == "prologue":
            c.update(rot=rot, fp32=fp32)
            cost = seq * c["heads"]
        elif op == "attention":
            c["entry"] = rng.choice(["strided", "strided", "head_major", "sdpa"])
            cost = int(_tile_mask(c).sum()) * c["heads"] if seq <= 33000 else 1 << 60
        elif op == "qkv":
            c.update(hidden=hidden, rot=rot, fp32=fp32)
            cost = seq * hidden * 3 * c["heads"] * D
        elif op == "out_proj":
            c.update(hidden=hidden)
            cost = seq * hidden * c["heads"] * D
        else:
            c.update(hidden=hidden, rot=rot, fp32=False,
                     projection=rng.choice(["fused", "hipblaslt"]))
            cost = seq * hidden * 4 * c["heads"] * D
            if seq <= 33000 and int(_tile_mask(c).sum()) * c["heads"] > 300_000:
                cost = 1 << 60
        if seq <= 33000 and cost <= _CAP[op]:
            return c


# ------------------------------------------------------------ shapes and masks

def _seq(c):
    return c["prefix"] + c["frames"] * c["height"] * c["width"]


def _tiles(c):
    return (_seq(c) + T - 1) // T


def _keyframes(c, seed):
    """What a plan's caller picks per render: two of the frames (two of the
    tile columns for a band) that every token attends to."""
    return sorted(random.Random(seed).sample(range(c["frames"]), 2))


def _landmarks(c):
    """First, middle and last frame: three landmarks evenly spaced."""
    last = c["frames"] - 1
    return sorted({0, last // 2 if last % 2 == 0 else (last + 1) // 2, last}) if last else [0]


def _rule(c, keys=None):
    s = _seq(c)
    if c["rule"] == "dense":
        return h3hip.MaskRule.dense(s)
    if c["rule"] == "band":
        return h3hip.MaskRule.band_rule(s, band=2, global_cols=tuple(keys or (0,)))
    if c["rule"] == "axial":
        return h3hip.MaskRule.axial(c["prefix"], c["frames"], c["height"], c["width"],
                                    landmarks=keys or _landmarks(c))
    return h3hip.MaskRule.local_window(c["prefix"], c["frames"], c["height"], c["width"],
                                       frame_window=1, spatial_tile=(8, 8), spatial_window=1,
                                       landmarks=tuple(keys or ()))


def _tile_mask(c, keys=None):
    """Active 128x128 tiles [n, n] bool, from the rule's written definition:
    tokens grouped into regions the rule cannot tell apart, a tile pair active
    when some region of one sees some region of the other."""
    n, prefix = _tiles(c), c["prefix"]
    if c["rule"] == "dense":
        return np.ones((n, n), bool)
    i = np.arange(n)
    if c["rule"] == "band":
        m = np.abs(i[:, None] - i[None, :]) <= 2
        m[:, keys or [0]] = True
        return m
    h, w, f = c["height"], c["width"], c["frames"]
    v = np.arange(f * h * w)
    fr, y, x = v // (h * w), v // w % h, v % w
    tile = (v + prefix) // T

    def incidence(region, count):
        a = np.zeros((n, count), np.float32)
        a[tile, region] = 1
        return a

    if c["rule"] == "local":
        ny, nx = (h + 7) // 8, (w + 7) // 8
        a = incidence((fr * ny + y // 8) * nx + x // 8, f * ny * nx)
        r = np.arange(f * ny * nx)
        rf, ry, rx = r // (ny * nx), r // nx % ny, r % nx
        g = ((np.abs(rf[:, None] - rf) <= 1) & (np.abs(ry[:, None] - ry) <= 1)
             & (np.abs(rx[:, None] - rx) <= 1) | np.isin(rf, keys or [])).astype(np.float32)
        m = a @ g @ a.T > 0
    else:
        a, p = incidence(fr, f), incidence(y * w + x, h * w)
        g = np.eye(f, dtype=np.float32)
        g[:, keys or _landmarks(c)] = 1
        m = (a @ g @ a.T > 0) | (p @ p.T > 0)
    if prefix:
        t = (prefix - 1) // T + 1
        m[:t] = m[:, :t] = True
    return m


# -------------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, shape, scale=1.0):
    return (torch.randn(shape, generator=g, device=DEV) * scale).to(torch.bfloat16)


def _gamma(g):
    return (0.9 + 0.2 * torch.rand(D, generator=g, device=DEV)).to(torch.bfloat16)


def _rope_inputs(c):
    """Positions (prefix at the origin, then the t, h, w lattice) and the pair
    tables of the case's rotary split, on the GPU."""
    s, p = _seq(c), c["prefix"]
    pos = torch.zeros((s, 3), device=DEV)
    v = torch.arange(s - p, device=DEV)
    h, w = c["height"], c["width"]
    pos[p:, 0], pos[p:, 1], pos[p:, 2] = v // (h * w), v // w % h, v % w
    axis, inv = [], []
    for a, d in enumerate(PAIR_DIMS[c["rot"]]):
        axis += [a] * (d // 2)
        inv += [10000.0 ** (-2.0 * k / d) for k in range(d // 2)]
    return (pos, torch.tensor(axis, dtype=torch.int32, device=DEV),
            torch.tensor(inv, dtype=torch.float32, device=DEV))


def _layer_inputs(c, seed):
    g, inner, hidden = _gen(seed), c["heads"] * D, c["hidden"]
    x = _randn(g, (_seq(c), hidden))
    wqkv = _randn(g, (3 * inner, hidden), 0.02)
    gq, gk = _gamma(g), _gamma(g)
    wout = _randn(g, (hidden, inner), 0.02) if c["op"] == "layer" else None
    return x, wqkv, gq, gk, wout


def _attention_inputs(c, seed):
    """q, k, v [H, S, D]: head-major storage padded to whole tiles, V or all
    three inside a token-major fused qkv for the entries that read it there."""
    g, H, s, n = _gen(seed), c["heads"], _seq(c), _tiles(c) * T
    if c["entry"] == "sdpa":
        qkv = _randn(g, (s, 3, H, D))
        return tuple(qkv[:, i].transpose(0, 1) for i in range(3))
    q, k = (_randn(g, (H, n, D)) for _ in range(2))
    if c["entry"] == "strided":
        return q[:, :s], k[:, :s], _randn(g, (s, 3, H, D))[:, 2].transpose(0, 1)
    return q, k, _randn(g, (H, n, D))


def _context(c):
    return AttentionContext(block_index=4, block_count=8, schedule_progress=0.5,
                            sequence_length=_seq(c))


def prepare(case, seed):
    c, st = case, {"case": case}
    op, H = c["op"], c["heads"]
    if op == "plan":
        st["rule"] = _rule(c, _keyframes(c, seed))
        st["cols"] = np.full(_tiles(c) ** 2, -1, np.int32)
    elif op == "prologue":
        g = _gen(seed)
        st["qkv"] = _randn(g, (_seq(c), 3 * H * D), 1.4)
        st["gammas"] = _gamma(g), _gamma(g)
        st["rope"] = _rope_inputs(c)
    elif op == "attention":
        st["plan"] = h3hip.TilePlan(_rule(c), heads=H)
        st["qkv"] = _attention_inputs(c, seed)
        st["backend"], st["context"] = H3HIPBackend(st["plan"]), _context(c)
    elif op == "out_proj":
        g = _gen(seed)
        st["x"] = _randn(g, (_seq(c), H * D), 0.3)
        st["w"] = _randn(g, (c["hidden"], H * D), 0.02)
    else:
        x, wqkv, gq, gk, wout = _layer_inputs(c, seed)
        mode = L.ROUND_FP32 if c["fp32"] else L.ROUND_REFERENCE
        st["x"] = x
        st["rope"] = RopeState.build(*_rope_inputs(c), rounding=mode)
        st["weights"] = wqkv, gq, gk
        if op == "layer":
            st["plan"] = h3hip.TilePlan(_rule(c), heads=H)
            st["context"] = _context(c)
            st["layer"] = AttentionLayer(wqkv, wout, gq, gk, heads=H, eps=EPS,
                                         backend=H3HIPBackend(st["plan"]),
                                         projection=c["projection"])
    return st


def run(state):
    c = state["case"]
    op, H = c["op"], c["heads"]
    if op == "plan":
        plan = h3hip.TilePlan(state["rule"], heads=H)
        row_ptr, cols = plan.tiles()
        plan.close()
        # The program's own list buffer, sized for any keyframes (unused: -1).
        state["cols"][:cols.size] = cols
        state["cols"][cols.size:] = -1
        return row_ptr, state["cols"]
    if op == "prologue":
        qkv, inner = state["qkv"], H * D
        pos, axis, inv = state["rope"]
        mode = L.ROUND_FP32 if c["fp32"] else L.ROUND_REFERENCE
        q, k, _ = ops.qk_norm_rope(qkv[:, :inner], qkv[:, inner:2 * inner], *state["gammas"], pos,
                                   axis, inv, heads=H, eps=EPS, rot=c["rot"], rounding=mode)
        return q, k
    if op == "attention":
        q, k, v = state["qkv"]
        if c["entry"] == "head_major":
            return ops.bsattn_fwd(state["plan"], q, k, v)
        if c["entry"] == "strided":
            return ops.bsattn_fwd_strided(state["plan"], q, k, v)
        return sdpa(*(t.transpose(0, 1) for t in (q, k, v)), D, backend=state["backend"],
                    context=state["context"])
    if op == "out_proj":
        return ops.out_proj(state["x"], state["w"])
    if op == "layer":
        return state["layer"](state["x"], state["rope"], state["context"])
    rope = state["rope"]
    return ops.qkv_proj(state["x"], *state["weights"], rope.table, heads=H, eps=EPS,
                        rounding=rope.rounding)


# ------------------------------------------------------- floors and tolerances

def work(case):
    c, H, s, n = case, case["heads"], _seq(case), _tiles(case)
    op, inner = c["op"], H * D
    pad = n * T
    nnz = int(_tile_mask(c).sum()) if op in ("plan", "attention", "layer") else 0
    attn_flops = 4.0 * T * T * D * nnz * H
    if op == "plan":      # the lists (without keyframes) and one schedule entry per (head, tile)
        return {"bytes": 4.0 * (n + 1 + nnz + H * n), "flops": 0.0}
    if op == "prologue":
        return {"bytes": 2.0 * 2 * inner * (s + pad) + 12.0 * s, "flops": 20.0 * inner * s}
    if op == "attention":
        return {"bytes": 4.0 * 2 * inner * s, "flops": attn_flops}
    hid = c["hidden"]
    if op == "out_proj":
        return {"bytes": 2.0 * (s * inner + hid * inner + s * hid), "flops": 2.0 * s * hid * inner}
    table = s * c["rot"] * 2 * (4.0 if c["fp32"] else 2.0)
    if op == "qkv":
        return {"bytes": 2.0 * (s * hid + 3 * inner * hid + 3 * inner * pad) + table,
                "flops": 2.0 * s * hid * 3 * inner}
    return {"bytes": 2.0 * (2 * s * hid + 4 * inner * hid) + table,
            "flops": 2.0 * s * hid * 4 * inner + attn_flops}


def tolerance(case):
    op = case["op"]
    if op == "plan":
        return "exact"
    if op == "prologue":
        return {"rel": 1.2e-2, "max": 6e-2}
    if op == "attention":
        return {"rel": 1e-2, "max": 6e-2}
    if op == "out_proj":
        return {"rel": 7e-3, "max": 3e-2}
    if op == "qkv":
        return {"rel": 1.2e-2, "max": 6e-2}
    return {"rel": 2e-2, "max": 1.2e-1}


# ----------------------------------------------------------------- in 64 bits

def _norm_rope64(x, gamma, rope, rot):
    """[S, H, D] float64 -> RMS norm, gamma, split-half rotation."""
    pos, axis, inv = rope
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gamma.double()
    ang = pos.double()[:, axis.long()] * inv.double()
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]
    a, b = y[..., :rot // 2], y[..., rot // 2:rot]
    return torch.cat([cos * a - sin * b, sin * a + cos * b, y[..., rot:]], dim=-1)


def _head_major64(x, pad):
    """[S, H, D] -> [H, pad, D], rows past S zero."""
    out = torch.zeros((x.shape[1], pad, D), dtype=torch.float64, device=x.device)
    out[:, :x.shape[0]] = x.transpose(0, 1)
    return out


def _attention64(c, q, k, v):
    """[H, S, D] of any dtype -> [H, S, D] float64 over the active tiles, one
    query tile of all heads at a time."""
    s = _seq(c)
    mask = torch.from_numpy(_tile_mask(c)).to(q.device)
    out = torch.zeros((c["heads"], s, D), dtype=torch.float64, device=q.device)
    for i in range(_tiles(c)):
        keys = mask[i].repeat_interleave(T)[:s].nonzero()[:, 0]
        rows = slice(i * T, min(s, (i + 1) * T))
        if keys.numel() == 0:
            continue
        kt = k[:, keys].double().transpose(1, 2).contiguous()
        p = torch.softmax(q[:, rows].double() @ kt / math.sqrt(D), dim=-1)
        out[:, rows] = p @ v[:, keys].double()
    return out


def exact(case, seed):
    c, op, H, s = case, case["op"], case["heads"], _seq(case)
    pad, inner = _tiles(c) * T, H * D
    if op == "plan":
        m = _tile_mask(c, _keyframes(c, seed))
        row_ptr = np.concatenate([[0], np.cumsum(m.sum(1))]).astype(np.int32)
        cols = np.full(m.size, -1, np.int32)
        cols[:m.sum()] = np.nonzero(m)[1]
        return row_ptr, cols
    if op == "prologue":
        g = _gen(seed)
        qkv = _randn(g, (s, 3 * inner), 1.4)
        gq, gk = _gamma(g), _gamma(g)
        rope = _rope_inputs(c)
        return tuple(_head_major64(_norm_rope64(
            qkv[:, i * inner:(i + 1) * inner].double().view(s, H, D), gam, rope, c["rot"]), pad)
            for i, gam in enumerate((gq, gk)))
    if op == "attention":
        q, k, v = _attention_inputs(c, seed)
        o = _attention64(c, q[:, :s], k[:, :s], v[:, :s])
        if c["entry"] == "head_major":
            return _head_major64(o.transpose(0, 1), pad)
        return o.transpose(0, 1).reshape(s, inner)
    if op == "out_proj":
        g = _gen(seed)
        x = _randn(g, (s, inner), 0.3)
        return x.double() @ _randn(g, (c["hidden"], inner), 0.02).double().t().contiguous()
    x, wqkv, gq, gk, wout = _layer_inputs(c, seed)
    rope = _rope_inputs(c)
    parts = []
    for i, gam in enumerate((gq, gk, None)):
        y = (x.double() @ wqkv[i * inner:(i + 1) * inner].double().t().contiguous()).view(s, H, D)
        parts.append(y if gam is None else _norm_rope64(y, gam, rope, c["rot"]))
    if op == "qkv":
        return tuple(_head_major64(y, pad) for y in parts)
    o = _attention64(c, *(y.transpose(0, 1) for y in parts))
    return o.transpose(0, 1).reshape(s, inner) @ wout.double().t().contiguous()
