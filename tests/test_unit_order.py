"""Work-group to unit arithmetic of the grouped GEMMs (exq_amd/csrc/unit_order.h), compiled for
the CPU: the ranges of the combined tile launch as its kernel walks them, and the order of the
rows kernels' units."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "exq_amd" / "csrc"

_SRC = r"""
#include "unit_order.h"
using namespace exq;
extern "C" {
int64_t t_unit_count(int64_t n, int n_tiles) { return unit_count(n, n_tiles); }
void t_mix(int t256, int t128, const int64_t* cap, int* tiles, int64_t* grid) {
  const MixTiles t = mix_tiles(t256, t128, cap[0], cap[1], cap[2], cap[3]);
  tiles[0] = t.ps; tiles[1] = t.i8; tiles[2] = t.t64; tiles[3] = t.bf;
  *grid = mix_grid(t, cap[0], cap[1], cap[2], cap[3]);
}
int t_rows_unit(int bid, int n, int n_tiles, int* tgi, int* nt) {
  return rows_unit_of(bid, n, n_tiles, *tgi, *nt);
}
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("unit_order")
    (d / "t.cpp").write_text(_SRC)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC",
                    f"-I{CSRC}", str(d / "t.cpp"), "-o", str(d / "t.so")], check=True)
    lb = C.CDLL(str(d / "t.so"))
    lb.t_unit_count.restype = C.c_int64
    lb.t_unit_count.argtypes = [C.c_int64, C.c_int]
    return lb


def _ranges(lib, t256, t128, caps, groups):
    """(grid, [units of each range as the kernel counts them]); groups: token groups of the list
    per range (128 x 256 INT4, INT8, 64 x 256 INT4, BF16)."""
    cap = (C.c_int64 * 4)(*caps)
    tiles, grid = (C.c_int * 4)(), C.c_int64()
    lib.t_mix(t256, t128, cap, tiles, C.byref(grid))
    return grid.value, [lib.t_unit_count(n, t) for n, t in zip(groups, tiles)]


@pytest.mark.parametrize("caps,groups", [
    # INT8 tiles beside INT4 experts on the grouped kernel (group sizes 256, 384, ...): the list's
    # INT4 groups are class 3 (no big experts) and no part of the launch
    ((0, 24, 0, 0), (0, 13, 45, 0)),
    ((0, 24, 0, 24), (0, 13, 45, 6)),
    ((0, 24, 0, 24), (0, 0, 45, 6)),
    # every tier on tiles: 64 x 256 tiles alone, with big experts, and scaled-operand tiles only
    ((0, 24, 90, 24), (0, 13, 45, 6)),
    ((20, 24, 90, 24), (7, 13, 45, 6)),
    ((90, 24, 0, 24), (45, 13, 0, 6)),
    ((0, 24, 0, 0), (0, 24, 0, 0)),
])
@pytest.mark.parametrize("t256,t128", [(1, 2), (8, 16), (11, 22)])
def test_mix_ranges_hold_only_launched_tiles(lib, caps, groups, t256, t128):
    grid, units = _ranges(lib, t256, t128, caps, groups)
    for cap, n, u in zip(caps, groups, units):
        if cap == 0:
            assert u == 0, "units of a range that the launch does not have"
        elif n:
            assert u > 0
    assert sum(units) <= grid, "the grid ends before the last unit"


@pytest.mark.parametrize("n_tiles", [1, 3, 16, 224])
@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 10, 11, 15, 16, 17, 24, 25, 31, 105])
def test_rows_units_once_each_and_even_over_the_xcds(lib, n, n_tiles):
    """Every unit is some work-group's (of a grid sized for n token groups or more), once, and no
    XCD (work-group number modulo 8) has more than an eighth of them, rounded up."""
    grid = 8 * -(-n // 8) * n_tiles
    tgi, nt = C.c_int(), C.c_int()
    seen, per_xcd = set(), [0] * 8
    for bid in range(grid + 8 * n_tiles):
        if lib.t_rows_unit(bid, n, n_tiles, C.byref(tgi), C.byref(nt)):
            assert bid < grid
            seen.add((tgi.value, nt.value))
            per_xcd[bid % 8] += 1
    assert seen == {(g, t) for g in range(n) for t in range(n_tiles)}
    assert sum(per_xcd) == n * n_tiles
    assert max(per_xcd) <= -(-n * n_tiles // 8)
