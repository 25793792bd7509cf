"""Code-generation properties the kernels' performance rests on, checked on the
CPU by compiling them to gfx950 assembly.

- bsattn_fwd.hip: the tile loop is one inline-assembly block with registers
  assigned by hand (bsattn_tile_loop.inc); the compiled kernel must carry all
  of its MFMAs, keep two waves per SIMD (at most 128 VGPRs and 128 AGPRs),
  and spill nothing to scratch around it (lane values are rebuilt per unit
  from an opaque thread index for that reason).
- bsattn_half.hip: the same of its tile loop (bsattn_half_loop.inc), one wave
  per SIMD.
- proj_gemm.hip: the reduction loops (gemm_loop.inc) are inline assembly with
  registers assigned by hand; every instantiation (nine tile shapes of four
  fused QKV forms, the plain QKV GEMM and the out-projection) must carry its
  shape's MFMAs and spill nothing, and keep one wave per SIMD (512 registers).
- qkv_proj.hip: no VGPR spills (scratch traffic) in any instantiation (the same
  six forms).

A different compiler release may allocate differently; a failure here says
to re-measure the kernel, not that its results are wrong.
"""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "minimax-h3-swift_amd", "csrc")


def _asm(tmp_path, name):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    out = tmp_path / (name + ".s")
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", f"-I{CSRC}", f"-I{os.path.join(ROOT, 'include')}",
                    "--cuda-device-only", "-S", "-o", str(out), os.path.join(CSRC, name + ".hip")],
                   check=True, capture_output=True)
    return out.read_text()


def _counts(asm, name):
    return [int(x) for x in re.findall(rf"\.{name}:\s+(\d+)", asm)]


def _mfmas(text, shape):
    return sum(1 for ln in text.splitlines() if ln.strip(' "').startswith("v_mfma_f32_" + shape))


@pytest.mark.parametrize("name,inc,registers", [
    ("bsattn_fwd", "bsattn_tile_loop", 256),     # two waves per SIMD
    ("bsattn_half", "bsattn_half_loop", 512),    # one
])
def test_attention_tile_loop_compiled_whole(tmp_path, name, inc, registers):
    asm = _asm(tmp_path, name)
    text = open(os.path.join(CSRC, inc + ".inc")).read()
    want = int(re.search(r"// \d+ lines, (\d+) MFMAs", text).group(1))
    n = _mfmas(asm, "32x32x16_bf16")
    assert n == want, (n, want)
    spills = _counts(asm, "vgpr_spill_count")
    assert spills and max(spills) == 0, spills
    scratch = _counts(asm, "private_segment_fixed_size")
    assert scratch and max(scratch) == 0, scratch
    agpr, vgpr = _counts(asm, "agpr_count"), _counts(asm, "vgpr_count")
    assert max(agpr) <= registers // 2 and max(vgpr) <= registers, (agpr, vgpr)


def test_projection_no_vgpr_spills(tmp_path):
    asm = _asm(tmp_path, "qkv_proj")
    spills = _counts(asm, "vgpr_spill_count")
    assert len(spills) == 6 and max(spills) == 0, spills


def test_four_wave_projection_compiled_whole(tmp_path):
    asm = _asm(tmp_path, "proj_gemm")
    inc = open(os.path.join(CSRC, "gemm_loop.inc")).read()
    forms = 6
    spills, scratch = _counts(asm, "vgpr_spill_count"), _counts(asm, "private_segment_fixed_size")
    assert len(spills) == len(scratch) == 9 * forms
    assert max(spills) == 0 and max(scratch) == 0, (spills, scratch)
    assert _mfmas(asm, "16x16x32_bf16") == forms * _mfmas(inc, "16x16x32_bf16")
    assert max(_counts(asm, "vgpr_count")) <= 512 and max(_counts(asm, "agpr_count")) <= 256
