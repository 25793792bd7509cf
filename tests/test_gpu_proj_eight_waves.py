"""The eight-wave projection kernel (qkv_proj_kernel), which short reductions over
more than one round of tiles run on: 1, 2, 3, 5 and 8 reduction steps, both
rotation widths and roundings, the plain GEMM and the out-projection, ragged
last tiles, a seq_pad that ends inside a token tile, and strided operands. All
sizes pick that kernel and their row subsets the four-wave one
(test_proj_tile_host.py holds both).

The plain GEMM is compared with an fp32 product on the CPU, each bf16 output
within half a bf16 ulp plus 1e-3 rms for the order of fp32 sums; the fused call
with h3hip_qk_norm_rope on the plain result, bit for bit; and rows of the plain
GEMM with the same rows as a call of their own on the four-wave kernel, bit for
bit: both add a channel's products in the same order."""
import pytest
import torch

from _gpu import bits, note
from test_gpu_out_proj import _check_fp32, _operands
from test_gpu_qkv_proj import _check_plain, _run

pytestmark = pytest.mark.gpu

ROWS = 100   # of a subset; 14 and 40 heads' worth of channels fit in one round then

# (S, hidden, H, rot, rounding, ldx, ldw)
QKV = [
    (2000, 320, 14, 128, 0, None, None),   # 8 x 21 tiles: lists of 24 and 20
    (2100, 128, 14, 96, 1, None, None),    # seq_pad 2,176 ends inside the ninth token tile
    (2050, 192, 14, 96, 0, None, None),    # two valid rows in the ninth
    (1000, 64, 40, 128, 1, None, None),    # one step
    (3000, 64, 14, 128, 0, 72, 88),
    (1100, 512, 40, 96, 1, 520, None),     # 5 x 60 tiles: full and short chunks on each XCD
]
# (S, in_features, out_features, ldx, ldw, ldy)
OUT = [
    (2000, 64, 5120, None, None, None), (2000, 128, 5120, None, None, 5128),
    (2049, 192, 5120, 200, 208, None),     # one valid row in the ninth token tile
    (2000, 320, 5120, None, None, None), (2000, 512, 5120, 520, None, 5136),
]


@pytest.mark.parametrize("S,hidden,H,rot,rounding,ldx,ldw", QKV)
def test_qkv(orc, S, hidden, H, rot, rounding, ldx, ldw):
    from h3hip import ops
    note(f"qkv eight waves S={S} hidden={hidden} H={H} rot={rot} rounding={rounding}")
    x, w, plain, fused, (want_q, want_k) = _run(orc, S, hidden, H, rot, rounding, ldx=ldx, ldw=ldw)
    _check_plain(*plain, x, w, S)
    assert torch.equal(fused[0], want_q) and torch.equal(fused[1], want_k)
    assert torch.equal(fused[2], plain[2])
    assert all((bits(t[:, S:]) == 0).all() for t in fused)
    for r in (0, S // 2, S - ROWS):
        part = ops.qkv_proj(x[r:r + ROWS], w, heads=H)
        torch.cuda.synchronize()
        for whole, rows in zip(plain, part):
            assert (bits(whole[:, r:r + ROWS]) == bits(rows[:, :ROWS])).all()


@pytest.mark.parametrize("S,fin,fout,ldx,ldw,ldy", OUT)
def test_out_proj(S, fin, fout, ldx, ldw, ldy):
    from h3hip import ops
    note(f"out_proj eight waves S={S} in={fin} out={fout} ldx={ldx} ldw={ldw} ldy={ldy}")
    x, w = _operands(S, fin, fout, 11, ldx, ldw)
    buf = torch.full((S + 2, ldy or fout), 7.0, dtype=torch.bfloat16, device="cuda")
    y = ops.out_proj(x, w, out=buf[:S, :fout])
    torch.cuda.synchronize()
    _check_fp32(y, x, w)
    assert torch.all(buf[S:] == 7.0) and torch.all(buf[:, fout:] == 7.0)
    for r in (0, S // 2, S - ROWS):
        part = ops.out_proj(x[r:r + ROWS], w)
        torch.cuda.synchronize()
        assert (bits(y[r:r + ROWS]) == bits(part)).all()
