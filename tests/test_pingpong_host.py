"""The index arithmetic of the dense product core (csrc/pingpong.hpp), enumerated on the host: a small program includes the
header the kernels include and calls the functions the kernels call."""
import os
import shutil
import subprocess

import pytest

from nanoquantization_amd import build as nq_build

PROGRAM = r"""
#include "pingpong.hpp"
#include <cstdio>
#include <vector>

static int fail(const char* what, int a, int b, int c, int d) {
    std::printf("%s: %d %d %d %d\n", what, a, b, c, d);
    return 1;
}

// Every tile is taken once, by grids that fit and by grids made for more tiles than there are.
static int tiles() {
    for (int x_tiles : {0, 1, 2, 7, 8, 9, 16, 17, 64, 68, 72, 128, 160})
        for (int w_tiles : {1, 2, 3, 8, 9, 48})
            for (int max_tiles : {x_tiles, x_tiles + 1, x_tiles + 4, x_tiles + 32, 160}) {
                if (max_tiles < x_tiles) continue;
                const int grid = (max_tiles * w_tiles + 7) / 8 * 8;
                std::vector<int> taken(x_tiles * w_tiles);
                for (int wg = 0; wg < grid; ++wg) {
                    int xt = -1, wt = -1;
                    if (!awq::xcd_tile(wg, x_tiles, w_tiles, xt, wt)) continue;
                    if (xt < 0 || xt >= x_tiles || wt < 0 || wt >= w_tiles) return fail("tile out of range", wg, xt, wt, grid);
                    ++taken[xt * w_tiles + wt];
                }
                for (int t = 0; t < x_tiles * w_tiles; ++t)
                    if (taken[t] != 1) return fail("tile not taken once", x_tiles, w_tiles, grid, taken[t]);
            }
    return 0;
}

// Every request of a tile, those for stages past the last one included, lies inside its operand: `rows` rows of `steps`
// stages, of which the tile begins at row `first` (the rows behind the last one come from it).
template <int XR>
static int requests() {
    using P = awq::PingPong<awq::BF16, XR>;
    for (int steps : {1, 2, 3, 5})
        for (int rows : {1, 2, 8, 31, XR - 1, XR, XR + 1, 3 * XR})
            for (int first = 0; first < rows; first += XR)
                for (int wave = 0; wave < 8; ++wave)
                    for (int lane = 0; lane < 64; ++lane)
                        for (int t = 0; t < steps + 2; ++t) {
                            const uint32_t row_bytes = steps * P::kStage * 2, size = rows * row_bytes;
                            const uint32_t stage = P::stage_bytes(t, steps);
                            if (t < steps && stage != (uint32_t)t * P::kStage * 2) return fail("wrong stage", t, steps, stage, XR);
                            for (int q = 0; q < 4; ++q) {
                                const int r = P::w_row(q, wave, lane);
                                const uint32_t at = P::source(first + r, rows, row_bytes, r, lane) + stage;
                                if (r < 0 || r >= P::kWR || at + 16 > size) return fail("weight request", rows, steps, t, at);
                            }
                            for (int q = 0; q < P::kXLoads; ++q) {
                                const int r = P::x_row(q, wave, lane);
                                const uint32_t at = P::source(first + r, rows, row_bytes, r, lane) + stage;
                                if (r < 0 || r >= XR || at + 16 > size) return fail("x request", rows, steps, t, at);
                            }
                        }
    return 0;
}

int main() { return tiles() || requests<128>() || requests<256>(); }
"""


@pytest.mark.skipif(shutil.which(nq_build.HIPCC) is None and not os.path.exists(nq_build.HIPCC), reason="hipcc not found")
def test_index_arithmetic_of_the_product_core(tmp_path):
    src, exe = tmp_path / "indices.hip", tmp_path / "indices"
    src.write_text(PROGRAM)
    built = subprocess.run([nq_build.HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17", f"-I{nq_build.CSRC}",
                            str(src), "-o", str(exe)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert built.returncode == 0, built.stdout[-2000:]
    ran = subprocess.run([str(exe)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert ran.returncode == 0, ran.stdout
