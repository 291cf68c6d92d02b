"""Tile addresses of the scatter P2G (gfsx_tiles.h) against Python's integers:
a tile's entries from its first one, on grids up to the 2^26 bricks that a step
takes, among them thin ones whose layers of entries together pass 2^32."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "gridfluidsim3d_amd", "csrc")

MAIN = r"""
#include "gfsx_tiles.h"
#include <cstdio>
int main() {
    long long base;
    int tx, ty, ex, ey, ez;
    unsigned x, y, z;
    while (scanf("%lld %d %d %d %d %d %u %u %u", &base, &tx, &ty, &ex, &ey, &ez, &x, &y, &z) == 9) {
        const gfsx::TileGrid t = {(size_t)base, tx, ty};
        printf("%zu\n", gfsx::tile_at(t, ex, ey, ez) + gfsx::tile_entry(t, x, y, z));
    }
}
"""


@pytest.mark.parametrize("bricks", [(1, 1, 1), (64, 64, 64), (5501, 5501, 1), (1, 5501, 5501),
                                    (8191, 8191, 1), (2, 2, 16777215), (67108863, 1, 1)])
def test_tile_entries(tmp_path, bricks):
    src, exe = tmp_path / "tiles.cpp", tmp_path / "tiles"
    src.write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    lines, want = [], []
    for c in range(3):
        size = [5 if a == c else 6 for a in range(3)]
        tx, ty = bricks[0] * size[0], bricks[1] * size[1]
        base = c * bricks[0] * bricks[1] * bricks[2] * 180
        for b in {(0, 0, 0), tuple(n - 1 for n in bricks), tuple(n // 2 for n in bricks)}:
            e = [b[a] * size[a] for a in range(3)]
            for i in {(0, 0, 0), (0, 0, size[2] - 1), tuple(n - 1 for n in size)}:
                lines.append("%d %d %d %d %d %d %d %d %d" % (base, tx, ty, *e, *i))
                want.append(base + e[0] + i[0] + tx * (e[1] + i[1] + ty * (e[2] + i[2])))
    out = subprocess.run([str(exe)], input="\n".join(lines), capture_output=True, text=True,
                         check=True).stdout.split()
    assert [int(v) for v in out] == want
