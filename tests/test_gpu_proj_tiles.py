"""proj_gemm_kernel's tile shapes where they can go wrong: one and few reduction
steps (rings not yet full), a step count that ends in every place of the
unrolled loop, a last tile of one row, padding rows past the last token tile,
strided operands. The sizes pick the tile they name (test_proj_tile_host.py).

The plain GEMM is compared with an fp32 product on the CPU, each bf16 output
within half a bf16 ulp plus 1e-3 rms for the order of fp32 sums
(|d| <= 2^-8 |want| + 1e-3 rms); the fused call with h3hip_qk_norm_rope on the
plain result, bit for bit."""
import pytest
import torch

from _gpu import bits, note
from test_gpu_out_proj import _check_fp32, _operands
from test_gpu_qkv_proj import _check_plain, _inputs, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile,S,fin,fout,ldx,ldy", [
    ("256x256", 1000, 1088, 15360, None, None),
    ("256x224", 801, 1024, 15360, None, None),
    ("256x192", 700, 1152, 15360, 1160, 15368),
    ("256x160", 600, 192, 15360, None, None),
    ("256x128", 1201, 192, 5120, 200, 5128),
    ("256x128", 1201, 64, 5120, None, None),
    ("256x128", 1160, 320, 5376, None, None),
    ("128x192", 1001, 192, 5120, None, None),
    ("128x160", 900, 320, 5120, None, 5128),
    ("128x128", 400, 448, 5120, 456, None),
    ("128x64", 129, 64, 256, None, 264),
])
def test_out_proj(tile, S, fin, fout, ldx, ldy):
    from h3hip import ops
    x, w = _operands(S, fin, fout, 11, ldx, ldx)
    note(f"out_proj tile {tile} S={S} in={fin} out={fout} ldx={ldx} ldy={ldy}")
    buf = torch.full((S + 2, ldy or fout), 7.0, dtype=torch.bfloat16, device="cuda")
    y = ops.out_proj(x, w, out=buf[:S, :fout])
    torch.cuda.synchronize()
    _check_fp32(y, x, w)
    assert torch.all(buf[S:] == 7.0) and torch.all(buf[:, fout:] == 7.0)


@pytest.mark.parametrize("tile,S,hidden,H,rot,rounding", [
    ("256x256", 1000, 1536, 40, 128, 0),
    ("256x224", 1270, 1600, 56, 96, 0),    # seq_pad 1,280 ends inside the sixth tile
    ("256x192", 1000, 1536, 56, 96, 1),    # seq_pad 1,024 ends inside the sixth tile
    ("256x160", 1100, 1536, 40, 128, 0),   # seq_pad 1,152 ends inside the eighth tile
    ("256x160", 600, 128, 40, 128, 1),
    ("256x128", 1250, 256, 14, 128, 0),
    ("128x192", 300, 704, 40, 128, 1),
    ("128x160", 800, 256, 14, 96, 0),      # seq_pad 896 ends inside the sixth tile
    ("128x128", 1000, 704, 6, 96, 0),
    ("128x64", 256, 64, 2, 96, 1),
] + [("128x64", 200, 64 * k, 2, 128, 0) for k in range(2, 8)])
def test_qkv(orc, tile, S, hidden, H, rot, rounding):
    note(f"qkv tile {tile} S={S} hidden={hidden} H={H} rot={rot} rounding={rounding}")
    x, w, plain, fused, (want_q, want_k) = _run(orc, S, hidden, H, rot, rounding)
    _check_plain(*plain, x, w, S)
    assert torch.equal(fused[0], want_q) and torch.equal(fused[1], want_k)
    assert torch.equal(fused[2], plain[2])


def test_padding_rows_past_the_last_token_tile():
    """seq_pad far past S: whole tiles, and the rest of a tile, of zero rows."""
    from h3hip import ops
    S, H, hidden = 130, 2, 128
    x, w = _inputs(S, hidden, H, 5)
    for seq_pad in (256, 384, 1024):
        note(f"qkv plain seq_pad={seq_pad}")
        out = [torch.full((H, seq_pad, 128), 7.0, dtype=torch.bfloat16, device="cuda")
               for _ in range(3)]
        ops.qkv_proj(x, w, heads=H, seq_pad=seq_pad, out=out)
        torch.cuda.synchronize()
        _check_plain(*out, x, w, S)
        assert all((bits(t[:, S:]) == 0).all() for t in out)


def test_more_token_tiles_than_a_signed_half_word():
    """32,770 token tiles of 256: rows on both sides of tile 32,768 and the last
    (a 1 GiB x; its one-step product keeps the run short)."""
    from h3hip import ops
    S, fin, fout = 32769 * 256 + 3, 64, 256
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    x = torch.empty((S, fin), dtype=torch.bfloat16, device="cuda").normal_(generator=g)
    w = torch.randn((fout, fin), generator=g, device="cuda").to(torch.bfloat16)
    note(f"out_proj S={S} in={fin} out={fout}")
    y = ops.out_proj(x, w)
    torch.cuda.synchronize()
    edge = 32768 * 256
    for r in (0, 1000, edge - 256, edge, edge + 255, S - 3):
        rows = slice(r, min(S, r + 256))
        _check_fp32(y[rows], x[rows], w)
