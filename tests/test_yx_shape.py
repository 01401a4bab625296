"""The shapes that yx_shape gives the fused y / x launch fit its LDS: where a
block's lanes evaluate its first x faces beforehand (64 columns), its rows
have a place in `first` (YxLds) and its waves one lane per row."""
from tests import hostprog

PROGRAM = r"""
#include "sonic_amd.h"
#include "sf_sweep.h"
#include <cstdio>
using namespace sfamd;
int main() {
    long long seen[2] = {0, 0};
    for (int cus : {8, 64, 256})
        for (int seg : {0, 1, 5, 32, 4096})
            for (int nx : {4, 31, 63, 64, 65, 127, 128, 190, 500, 853, 2048, 30000})
                for (int ny : {4, 33, 64, 97, 500, 853, 2048, 30000})
                    for (int nz : {1, 5, 64, 300}) {
                        if ((long long)nx * ny * nz > 1LL << 30) continue;
                        SweepCall c{};
                        const int n[3] = {nx, ny, nz};
                        for (int a = 0; a < 3; ++a) {
                            c.G.n[a] = n[a];
                            c.G.active[a] = n[a] > 1;
                            c.G.g[a] = n[a] > 1 ? 3 : 0;
                            c.G.solved_hi[a] = n[a] - 1;
                        }
                        c.A.time = 1;
                        c.seg = seg;
                        c.cus = cus;
                        c.x_walk = -1;
                        const YxShape sh = yx_shape(c);
                        if (!sh.blocks || sh.block) continue;
                        const int room = sh.waves > 1 ? YxLds<0, kYxWaves>::rows : YxLds<0, 1>::rows;
                        ++seen[sh.waves > 1];
                        const bool ok = sh.rows >= 1 && sh.rows <= kYxRows &&
                                        (sh.cols == kXBlock - 1 || (sh.cols == kXBlock && sh.rows <= room)) &&
                                        (long long)sh.nx * sh.cols >= nx &&
                                        (long long)sh.ny * sh.rows * sh.waves >= ny;
                        if (!ok) printf("%d x %d x %d seg %d: %d cols %d rows %d waves\n", nx, ny, nz, seg,
                                        sh.cols, sh.rows, sh.waves);
                    }
    printf("%s\n", seen[0] && seen[1] ? "done" : "no shapes");
}
"""


def test_shapes_fit_the_lds(tmp_path):
    assert hostprog.run(tmp_path, PROGRAM) == ["done"]
