"""The schedule a plan runs (plan_schedule in csrc/schedule.cpp, compiled here with
g++): whole units or half units, every one of them listed exactly once, one a
workgroup while there are no more half units than workgroups, and the unit size
that the GPU tests' plans are meant to have."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

import test_gpu_half_units as half_units

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "minimax-h3-swift_amd", "csrc")
GROUPS = 256

HARNESS = r"""
#include "schedule.cpp"
namespace h3hip {
void set_error(const char*, ...) {}
}
// 1 for half units, 0 for whole ones, negative for an error.
extern "C" int lists(const int32_t* row_ptr, int32_t n, int32_t heads, int32_t groups,
                     int32_t* work_ptr, int32_t* work) {
  std::vector<int32_t> rp(row_ptr, row_ptr + n + 1), wp, w;
  bool half = false;
  const int rc = h3hip::plan_schedule(rp, heads, groups, half, wp, w);
  if (rc) return rc;
  std::copy(wp.begin(), wp.end(), work_ptr);
  std::copy(w.begin(), w.end(), work);
  return half;
}
// Whether the plan's own check takes these units.
extern "C" int units_once(const int32_t* work, int32_t count, int32_t heads, int32_t rows) {
  return h3hip::check_units(heads, rows, std::vector<int32_t>(work, work + count)) == H3HIP_OK;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("schedule")
    (d / "h.cpp").write_text(HARNESS)
    subprocess.run([cxx, "-O1", "-std=c++17", "-fPIC", "-shared", "-I", CSRC, str(d / "h.cpp"),
                    "-o", str(d / "h.so")], check=True)
    return ctypes.CDLL(str(d / "h.so"))


def _p(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_int32))


def plan_lists(lib, lengths, heads, groups=GROUPS):
    """(unit_rows, work_ptr, work) of rows of these lengths."""
    rp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    n = len(lengths)
    work_ptr, work = np.zeros(groups + 1, np.int32), np.zeros(2 * heads * n, np.int32)
    half = lib.lists(_p(rp), n, heads, groups, _p(work_ptr), _p(work))
    assert half in (0, 1)
    return (64 if half else 128), work_ptr, work[:heads * n * (1 + half)]


def check_once(unit_rows, work_ptr, work, n, heads, groups=GROUPS):
    rows = n * 128 // unit_rows
    assert work_ptr[0] == 0 and work_ptr[-1] == len(work) == heads * rows
    assert np.all(np.diff(work_ptr) >= 0)
    ids = np.sort((work >> 16).astype(np.int64) * rows + (work & 0xFFFF))
    assert np.array_equal(ids, np.arange(heads * rows))
    if unit_rows == 64 and heads * rows <= groups:
        assert np.diff(work_ptr).max() == 1


@pytest.mark.parametrize("S,heads,kind,unit_rows", half_units.CASES)
def test_unit_size_of_the_gpu_cases(lib, S, heads, kind, unit_rows):
    n = (S + 127) // 128
    lengths = half_units._bitmap(kind, n, np.random.default_rng(S)).sum(1)
    got = plan_lists(lib, lengths, heads)
    assert got[0] == unit_rows
    check_once(*got, n, heads)
    if kind == "gaps":   # units without a tile before and after units with tiles
        _, work_ptr, work = got
        empty = lengths[(work & 0xFFFF) // 2] == 0
        pairs = {(bool(a), bool(b)) for i in range(GROUPS)
                 for a, b in zip(empty[work_ptr[i]:work_ptr[i + 1]],
                                 empty[work_ptr[i] + 1:work_ptr[i + 1]])}
        assert {(True, False), (False, True)} <= pairs


@pytest.mark.parametrize("S,heads,more,kind", half_units.PAIRS)
def test_unit_size_of_the_compared_plans(lib, S, heads, more, kind):
    n = (S + 127) // 128
    lengths = half_units._bitmap(kind, n, np.random.default_rng(S)).sum(1)
    assert plan_lists(lib, lengths, heads)[0] == 64
    assert plan_lists(lib, lengths, more)[0] == 128


@pytest.mark.parametrize("groups", [8, 64, 256, 304])
def test_every_unit_once(lib, groups):
    """Row counts and heads over both unit sizes, up to and past the last plan of
    one half unit per workgroup; empty, short and full rows."""
    rng = np.random.default_rng(groups)
    seen = set()
    for n, heads in [(1, 1), (1, groups // 2), (1, groups // 2 + 1), (3, 2), (7, 5), (13, 3),
                     (50, 2), (61, 30), (groups // 2, 1), (groups // 2 + 1, 1)]:
        for lengths in (np.full(n, n), rng.integers(0, n + 1, n), np.zeros(n, int),
                        np.where(np.arange(n) == n // 2, n, 1)):
            got = plan_lists(lib, lengths, heads, groups)
            seen.add(got[0])
            check_once(*got, n, heads, groups)
    assert seen == {64, 128}


def test_more_units_than_six_a_workgroup_stay_whole(lib):
    """Past that the GPU tests of whole units rely on whole units, whatever the rows."""
    for n, heads in [(1, 1537), (2, 769), (12, 129)]:
        for lengths in (np.full(n, n), np.where(np.arange(n) == 0, n, 0)):
            assert plan_lists(lib, lengths, heads)[0] == 128


def test_a_dropped_and_a_doubled_unit_are_refused(lib):
    work = np.array([0, 1, 2, 1 << 16, 1 << 16 | 1, 1 << 16 | 2], np.int32)
    assert lib.units_once(_p(work), 6, 2, 3) == 1
    assert lib.units_once(_p(work), 5, 2, 3) == 0
    work[5] = 0
    assert lib.units_once(_p(work), 6, 2, 3) == 0


def test_no_plan_is_refused(h3):
    from h3hip import _lib
    assert h3.lib().h3hip_plan_schedule(None, None, None, None, None) == _lib.EINVAL
    assert "plan is NULL" in h3.last_error()
