"""Host-side check of the bounds-checked result stores of the GEMM kernels: for sub-tiles over the last
columns of matrices up to several times 2 GiB, a store must be in range exactly when its row and its columns
lie inside the matrix, and must then address its own element. The offsets are those of
csrc/store_window.h, compiled here for the host and walked lane by lane as the kernels' epilogue does."""

import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "primus-turbo_amd" / "csrc"

PROGRAM = r"""
#include "store_window.h"
#include <cstdio>
#include <cstdlib>
using namespace pt;

// one sub-tile of `groups` x 16 rows and `width` columns at (wm, wn) of an [m, n] matrix
static long walk(int64_t m, int64_t n, int es, int64_t wm, int64_t wn, int groups, int width) {
    const uint32_t rb = static_cast<uint32_t>(n * es), row16 = 16 * rb;
    const int      cols = static_cast<int>(n - wn < width ? n - wn : width);
    const int      step = es == 4 ? 16 : 32;
    uint32_t       left = window_bytes(m, wm, wn, n, es);
    int64_t        base = (wm * n + wn) * es;
    long           bad  = 0;
    for (int i = 0; i < groups; ++i) {
        for (int lane = 0; lane < 64; ++lane) {
            const int      lm = lane & 15, lg = lane >> 4;
            const int      c0   = es == 4 ? 4 * lg : 16 * (lg & 1) + 8 * (lg >> 1);
            const uint32_t off0 = lm * rb + c0 * es;
            for (int j = 0; j < width / step; ++j) {
                const uint32_t off    = window_offset(off0, c0 + j * step, cols, 64 * j);
                const bool     stored = off < left; // (the bounds check of a buffer store)
                const int64_t  row = wm + 16 * i + lm, col = wn + c0 + j * step;
                const bool     want = row < m && col < n;
                const bool     fits = !stored || off + 16u <= left;
                if (stored != want || !fits || (stored && base + off != (row * n + col) * es))
                    ++bad;
            }
        }
        base += row16;
        left = window_next(left, row16);
    }
    return bad;
}

int main(int argc, char **argv) {
    const int64_t m = atoll(argv[1]), n = atoll(argv[2]);
    const int     es = atoi(argv[3]), tile = atoi(argv[4]), half = tile / 2;
    long          bad = 0, tiles = 0;
    // the sub-tiles of the last column of tiles: at the start, around 2 and 4 GiB from the end, and at the end
    const int64_t ends[] = {0, m - (int64_t{1} << 31) / (n * es), m - (int64_t{1} << 32) / (n * es), m};
    for (int64_t e : ends)
        for (int64_t wm = (e / half - 2) * half; wm <= (e / half + 1) * half; wm += half) {
            if (wm < 0 || wm / tile * tile >= m)
                continue;
            for (int64_t wn = (n - 1) / tile * tile; wn < (n - 1) / tile * tile + tile; wn += half) {
                bad += walk(m, n, es, wm, wn, half / 16, half);
                ++tiles;
            }
        }
    printf("%ld %ld\n", tiles, bad);
    return 0;
}
"""


@pytest.fixture(scope="module")
def walker(tmp_path_factory):
    d = tmp_path_factory.mktemp("window")
    (d / "w.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-I", str(CSRC), str(d / "w.cpp"), "-o", str(d / "w")], check=True)
    return d / "w"


@pytest.mark.parametrize("tile", [128, 256])
@pytest.mark.parametrize("es", [2, 4])
@pytest.mark.parametrize("m,n", [
    (1, 8), (333, 264), (3001, 2880),       # well below 2 GiB
    (8192, 151936),                         # 2.5 GB in 16 bits
    (70001, 16392), (262144, 8200),         # 2 to 8 GiB, eight columns in the last tile
    (1 << 21, 2056), (300, (1 << 22) - 8),  # rows at the widest
])
def test_stores_land_on_their_own_element(walker, m, n, es, tile):
    tiles, bad = map(int, subprocess.run([walker, str(m), str(n), str(es), str(tile)], capture_output=True, text=True,
                                         check=True).stdout.split())
    assert tiles > 0 and bad == 0, f"{bad} stores of {tiles} sub-tiles"
