"""Tiling of the environment projection at the map sizes it accepts (fewer than 2^31 cells), compiled on the
host under the undefined-behaviour sanitizer: the blocks' tiles cover the map once and no index
overflows."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include "env_tiles.h"
#include <cstdio>
#include <cstdlib>
using namespace bsh;
int main(int, char** argv)
{
    const int W = std::atoi(argv[1]), H = std::atoi(argv[2]);
    const EnvTiles t = env_tiles(W, H);
    const uint32_t n = (uint32_t)t.nx * (uint32_t)t.ny, step = n > 100000 ? n / 50000 : 1;
    std::printf("%d %d %d %d\n", t.cols, t.rows, t.nx, t.ny);
    for (uint32_t b = 0; b < n; b += (b + 2000 > n || b < 2000) ? 1 : step)
    {
        const EnvTile k = env_tile(b, t, H);
        std::printf("%u %d %d %d\n", b, k.col0, k.row0, k.row1);
    }
}
"""
LAST = (1 << 31) - 1


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("tiles")
    (d / "t.cpp").write_text(PROGRAM)
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=undefined", "-fno-sanitize-recover=all", "-I",
                        os.path.join(ROOT, "banshee_amd", "csrc"), str(d / "t.cpp"), "-o", str(d / "t")],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return str(d / "t")


@pytest.mark.parametrize("w,h", [(1, 1), (1, 700), (3, 5), (255, 2), (257, 129), (513, 517), (2048, 1024), (1, LAST),
                                 (1, LAST - 255), (2, LAST // 2), (300, LAST // 300), (46340, 46340), (LAST // 2, 2),
                                 (LAST - 200, 1), (LAST, 1)])
def test_tiles_cover_the_map(exe, w, h):
    r = subprocess.run([exe, str(w), str(h)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    rows = [tuple(map(int, ln.split())) for ln in r.stdout.splitlines()]
    (cols, per, nx, ny), tiles = rows[0], rows[1:]
    assert 1 <= cols <= 256 and 256 // cols <= per <= 256
    assert (nx - 1) * cols < w <= nx * cols and (ny - 1) * per < h <= ny * per
    for b, col0, row0, row1 in tiles:
        assert (col0, row0, row1) == (b % nx * cols, b // nx * per, min(b // nx * per + per, h))
    assert tiles[0][0] == 0 and tiles[-1][0] == nx * ny - 1
