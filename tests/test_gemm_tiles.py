"""Size and order of the GEMM's output tiles (csrc/gemm_tiles.h, compiled here as host code)."""
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
namespace mxf8 {
constexpr int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }
constexpr int GEMM_BK = 128;
}
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


# (M, N, K, LoRA rank): us of tiles 0-5 (gemm_pick) on MI355X, weights from HBM; None: not timed
TIMES = {
    (1, 3072, 3072, 0): (8.2, 10.0, 10.8, 14.6, 17.0, 30.9),
    (512, 3072, 3072, 0): (22.5, 12.6, 11.9, 15.8, 19.1, 32.6),
    (344, 6144, 2048, 0): (None, 17.5, 14.7, 13.8, 18.7, None),
    (512, 3072, 12288, 0): (74.0, 59.7, 52.1, 65.1, 110.2, 152.0),
    (1024, 3072, 12288, 0): (143.3, 82.8, 91.1, 65.5, 105.2, 149.5),
    (2048, 3072, 3072, 0): (83.6, 35.5, 28.0, 32.4, 23.8, 34.3),
    (20000, 192, 3072, 0): (55.7, 25.5, 19.6, 31.5, 23.1, 38.7),      # many more tokens than channels
    (16384, 256, 1024, 0): (28.6, 12.4, 9.6, 9.8, 9.4, 15.2),
    (4096, 1024, 2048, 0): (42.2, 18.5, 13.8, 13.7, 14.3, 24.3),
    (1024, 9216, 3072, 0): (137.3, 58.5, 48.1, 54.8, 54.4, 38.4),     # one round of 256 x 256
    (3072, 3072, 12288, 0): (395.0, 206.7, 181.5, 164.9, 183.6, 148.4),
    (1024, 3072, 3072, 128): (53.4, 27.3, 24.1, 24.7, 23.0, 38.2),
    (3072, 3072, 3072, 128): (None, None, 59.1, 70.6, 47.9, 41.9),
    (3072, 3072, 3072, 512): (None, None, 107.7, 131.5, 129.3, 145.8),  # a LoRA read from global memory
    (1536, 3072, 3072, 1024): (None, None, 110.6, 143.2, 134.4, 255.9),
    (2048, 3072, 3072, 2048): (None, None, 198.2, 256.8, 249.2, 486.6),
    (512, 6144, 1536, 4096): (295.3, 229.4, 236.7, 237.0, 268.9, 920.7),
    (4096, 3072, 12288, 256): (None, None, 278.0, 232.1, 274.4, 203.8),
}


@pytest.fixture(scope="module")
def pick(tmp_path_factory):
    """(M, N, K, r) -> the tile gemm_pick takes on 256 CUs."""
    run = host_program(tmp_path_factory.mktemp("pick"), """
int main() {
  long m, n, k, r;
  while (std::scanf("%ld %ld %ld %ld", &m, &n, &k, &r) == 4)
    std::printf("%d\\n", mxf8::gemm_pick(m, n, k, r, 256));
}""")
    return lambda *shape: run([shape])[0][0]


@pytest.mark.parametrize("shape", TIMES)
def test_pick_is_near_the_best_measured_tile(pick, shape):
    """Within a twelfth of the best tile, and never slower than the 128 x 128 tiles by more than the
    estimates are off."""
    times = TIMES[shape]
    t = times[pick(*shape)]
    assert t is not None
    assert t <= 1.08 * min(x for x in times if x is not None)
    assert t <= 1.03 * times[4]


@pytest.mark.parametrize("shape", [(20280, 9216, 3072, 0), (20280, 3072, 12288, 0), (77648, 9216, 3072, 64),
                                   (77648, 3072, 3072, 4096), (8192, 4096, 512, 0)])
def test_512_tiles_of_256_always_take_them(pick, shape):
    assert pick(*shape) == 5


@pytest.mark.parametrize("ring,fits", [("32, 64, 1, 2, 4, 2", True), ("32, 64, 1, 1, 4, 2", False)])
def test_ring_depth_is_bounded_by_the_copy_counter(ring, fits):
    """The first stage is waited for with NS - 1 later stages' copies in flight, and the counter
    holds 63: 36 of them, and 72 with one wave, which must not compile."""
    code = f'#include "gemm.hip"\nstatic_assert(mxf8::GemmRing<{ring}>::NS == 4, "");\n'
    res = subprocess.run([build.hipcc(), "--offload-arch=gfx950", "--offload-host-only", "-std=c++17", "-fsyntax-only",
                          "-I", build.CSRC, "-x", "hip", "-"], input=code, capture_output=True, text=True)
    assert (res.returncode == 0) == fits, res.stderr[-2000:]
    assert fits or "counts the copies" in res.stderr


# (N, K, LoRA rank): tokens that take tiles 0 to 5 (test_gpu_gemm_ring.py compares their bits)
EVERY_TILE = {
    (3072, 2064, 0): (33, 201, 401, 701, 1301, 2701),
    (2056, 3088, 32): (1, 299, 450, 1001, 2001, 4001),
    (3072, 6160, 48): (1, 170, 331, 700, 1401, 2701),
    (3072, 6160, 160): (1, 170, 331, 700, 1401, 2701),
}


@pytest.mark.parametrize("shape", EVERY_TILE)
def test_every_tile_is_compared(pick, shape):
    N, K, r = shape
    assert [pick(m, N, K, r) for m in EVERY_TILE[shape]] == [0, 1, 2, 3, 4, 5]
