"""How the register-resident kernel's workgroups share its units (csrc/unit_runs.h, compiled for the host): CPU tests."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "unit_runs.h"
extern "C" int first(int rows, int chunks, int columns, int chunk, int last, int b, int grid)
{
    return tship::UnitRuns{rows, chunks, columns, chunk, last}.first(b, grid);
}
extern "C" long long longest(int rows, int chunks, int columns, int chunk, int last, int grid, int kt, int unit, int cross)
{
    return tship::UnitRuns{rows, chunks, columns, chunk, last}.longest(grid, 4 * (chunk - 1), 4 * (last - 1), kt, unit, cross);
}
"""


@pytest.fixture(scope="module")
def first(tmp_path_factory):
    out = tmp_path_factory.mktemp("runs")
    (out / "runs.cpp").write_text(SOURCE)
    lib = str(out / "libruns.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I" + os.path.join(ROOT, "tensorsharp_amd", "csrc"), str(out / "runs.cpp"), "-o", lib], check=True)
    got = C.CDLL(lib)
    got.longest.restype = C.c_longlong
    got.first.longest = got.longest
    return got.first


# (row tiles, K chunks, column tiles, weight of a unit of a whole chunk, of the last chunk)
CASES = [(1, 1, 1, 5, 5), (1, 3, 4, 5, 3), (1, 5, 50, 3, 2), (2, 2, 16, 3, 2), (3, 4, 21, 5, 2), (1, 4, 64, 3, 2), (1, 4, 65, 3, 2), (1, 2, 300, 5, 2), (7, 3, 1344, 5, 3),
         (0, 2, 100, 3, 2), (2000, 8, 1344, 5, 2)]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("grid", [1, 12, 255, 256])
def test_every_unit_is_taken_once_and_in_order(first, case, grid):
    at = [first(*case, b, grid) for b in range(grid + 1)]
    assert at[0] == 0 and at[-1] == case[0] * case[1] * case[2] and at == sorted(at)


@pytest.mark.parametrize("case", [c for c in CASES if c[0] * c[1] * c[2] <= 256])
def test_a_workgroup_for_every_unit_takes_one(first, case):
    # two units of two chunks in one workgroup, next to workgroups with none, doubled the time of such launches
    units = case[0] * case[1] * case[2]
    for grid in (units, 256):
        assert all(first(*case, b + 1, grid) - first(*case, b, grid) == (b < units) for b in range(grid))


@pytest.mark.parametrize("case", [c for c in CASES if c[0] * c[1] * c[2] > 256])
def test_runs_weigh_about_the_same(first, case):
    rows, chunks, columns, chunk, last = case
    per = chunks * columns
    weigh = lambda u: last if u % per >= (chunks - 1) * columns else chunk
    total = rows * ((chunks - 1) * columns * chunk + columns * last)
    runs = [(first(*case, b, 256), first(*case, b + 1, 256)) for b in range(256)]
    if total < 10 ** 6:
        assert max(sum(weigh(u) for u in range(*r)) for r in runs) <= total / 256 + chunk


@pytest.mark.parametrize("case", [c for c in CASES if 0 < c[0] * c[1] * c[2] < 10 ** 5] + [(2, 2, 147, 3, 2), (1, 4, 256, 3, 2), (3, 1, 418, 3, 3), (5, 7, 33, 4, 2)])
@pytest.mark.parametrize("kt,unit,cross", [(19, 69, 240), (12, 67, 120), (1, 0, 0)])
def test_the_longest_run(first, case, kt, unit, cross):
    """Against all runs, where every edge is looked at: no run costs more, and what is said is at most one unit above the one that does most."""
    rows, chunks, columns, chunk, last = case
    cost = lambda u: kt * 4 * ((last if u // columns % chunks == chunks - 1 else chunk) - 1) + unit
    runs = [range(first(*case, b, 256), first(*case, b + 1, 256)) for b in range(256)]
    most = max(sum(map(cost, r)) + cross * (r[-1] // columns - r[0] // columns) for r in runs if len(r))
    got = first.longest(*case, 256, kt, unit, cross)
    assert got <= most + kt * 4 * (chunk - 1) + unit
    if rows * chunks <= 13:
        assert got >= most
