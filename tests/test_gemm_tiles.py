"""Order of the GEMM's output tiles (csrc/gemm_tiles.h, compiled here as host code)."""
import subprocess

import pytest

from minimaxh3_amd import build

# what the header takes from the HIP headers and the sources that include it
PRELUDE = """
#include <algorithm>
#include <cstdint>
#include <cstdio>
#define __host__
#define __device__
using std::max;
using std::min;
"""


def host_program(tmp_path, body):
    """Compile body after the header and return a function that runs it on lines of integers."""
    src, exe = tmp_path / "main.cpp", tmp_path / "main"
    src.write_text(f'{PRELUDE}\n#include "gemm_tiles.h"\n{body}')
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-Wno-unused-function", "-I", build.CSRC, str(src),
                    "-o", str(exe)], check=True)

    def run(lines):
        text = "".join(" ".join(map(str, line)) + "\n" for line in lines)
        out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    return run


@pytest.fixture(scope="module")
def ring_tiles(tmp_path_factory):
    """(tiles_m, tiles_n) -> the (XCD, token-tile, channel-tile) of every workgroup of the ring kernel."""
    run = host_program(tmp_path_factory.mktemp("tiles"), """
int main() {
  int m, n;
  while (std::scanf("%d %d", &m, &n) == 2)
    for (int s = 0; s < m * n; ++s) {
      int tm, tn;
      mxf8::tile_coords(s, m, n, mxf8::RING_GROUP_M, tm, tn);
      std::printf("%d %d %d\\n", s % 8, tm, tn);
    }
}""")
    return lambda m, n: run([(m, n)])


@pytest.mark.parametrize("m,n", [(1, 1), (1, 48), (8, 24), (9, 7), (150, 3), (128, 2), (64, 7), (32, 8), (48, 5),
                                 (3, 100)])
def test_ring_tiles_are_covered_once_and_share_panels(ring_tiles, m, n):
    """Each XCD runs an eighth of the tiles, in a block of few operand panels: it reads no more
    activation panels than rows of tiles that hold its share (and a group of 8 at either end),
    nor, up to 8 token-tiles, more weight panels than columns that hold it (and one)."""
    tiles = ring_tiles(m, n)
    assert sorted(t[1:] for t in tiles) == [(i, j) for i in range(m) for j in range(n)]
    for xcd in range(8):
        mine = [t for t in tiles if t[0] == xcd]
        assert len({t[1] for t in mine}) <= -(-len(mine) // n) + 16
        if m <= 8:
            assert len({t[2] for t in mine}) <= -(-len(mine) // m) + 1
