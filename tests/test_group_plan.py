"""How the grid form's workgroups of four row blocks cut their column ranges (csrc/km_group_plan.h, compiled for the
host): every column of a range is counted once for its row block, and none outside it."""
import ctypes
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "kernel_matmul_amd", "csrc")
SOURCE = """
#include "km_group_plan.h"
// ranges: four starts, four ends.  out: start, end and rows of the ten segments and the four pieces, whether the core
// is shared.
extern "C" void plan(const int* ranges, const int* sorted, int* out) {
    using namespace km;
    int ends[8], at[8];
    for (int i = 0; i < 8; i++) {
        ends[i] = ranges[i];
        at[i] = sorted[i];
    }
    const GroupCut c = group_cut(at);
    for (int i = 0; i < KM_GROUP_SEGMENTS + KM_GROUP; i++) {
        const bool piece = i >= KM_GROUP_PIECE;
        const int* bound = piece ? c.piece + i - KM_GROUP_PIECE : c.segment + i;
        out[3 * i] = bound[0];
        out[3 * i + 1] = bound[1];
        out[3 * i + 2] = group_rows(ends, bound[0], bound[1]);
    }
    out[3 * (KM_GROUP_SEGMENTS + KM_GROUP)] = c.shared;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    folder = tmp_path_factory.mktemp("plan")
    source, library = folder / "plan.cpp", folder / "plan.so"
    source.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{CSRC}", str(source), "-o", str(library)], check=True)
    function = ctypes.CDLL(str(library)).plan

    def call(ranges):
        """(start, end, rows) of the segments whose sums are added; the pieces of a shared core stand for it."""
        first = ranges[0][0]
        starts = [s if e > s else first for s, e in ranges]
        ends = [e if e > s else first for s, e in ranges]
        ends[0] = max(ranges[0])
        out = (ctypes.c_int * 43)()
        function((ctypes.c_int * 8)(*starts, *ends), (ctypes.c_int * 8)(*sorted(starts + ends)), out)
        cut = [tuple(out[3 * i:3 * i + 3]) for i in range(14)]
        shared = out[42]
        if shared:
            core = cut[4]
            assert cut[5][0] == cut[5][1]
            assert all(core[0] <= s <= e <= core[1] and rows in (0, core[2]) for s, e, rows in cut[10:])
            cut[4:5] = cut[10:]
        return cut[:-4]

    return call


def _check(plan, ranges):
    cells = [c for c in plan(ranges) if c[2]]
    lo, hi = min(s for s, _ in ranges), max(e for _, e in ranges)
    for row, (start, end) in enumerate(ranges):
        mine = sorted((s, e) for s, e, rows in cells if rows >> row & 1)
        if end <= start:
            assert not mine
            continue
        assert mine[0][0] == start and mine[-1][1] == end
        assert all(a[1] == b[0] for a, b in zip(mine, mine[1:]))
    # (what is read lies in the matrix, that of segments without columns too)
    assert all(lo <= s <= e <= hi for s, e, _ in plan(ranges))


@pytest.mark.parametrize("before,after", [
    ((0, 0, 0), (0, 0, 0)), ((128, 128, 128), (0, 0, 0)), ((0, 0, 0), (128, 128, 128)),
    ((128, 128, 128), (128, 128, 128)), ((119, 97, 140), (119, 116, 140)), ((1, 0, 31), (33, 1, 64)), ((0, 700, 3), (5, 0, 900)),
])
def test_every_width_of_the_shared_columns(plan, before, after):
    """Starts and ends so far apart, from row block to row block; the last range ends with the matrix."""
    for core in range(3001):
        starts = [7, 7 + before[0], 7 + sum(before[:2]), 7 + sum(before)]
        end = starts[3] + core
        ends = [end, end + after[0], end + sum(after[:2]), end + sum(after)]
        _check(plan, list(zip(starts, ends)))
        _check(plan, [(s, ends[3]) for s in starts])


def test_ranges_that_lie_anywhere(plan):
    g = random.Random(1)
    for _ in range(20_000):
        width = g.choice([40, 300, 900, 3000])
        ranges = [(g.randrange(width), g.randrange(width)) for _ in range(4)]
        _check(plan, [(s, max(s, e)) for s, e in ranges])


def test_ranges_at_the_largest_size(plan):
    n = 2**31 - 1 - 128
    for ranges in ([(0, n)] * 4, [(n, n), (n - 1, n), (n - 40, n), (0, n)], [(n - 300, n)] * 4, [(0, 5), (n - 5, n), (3, 3), (n - 3, n - 1)]):
        _check(plan, ranges)
