"""The 32-bit byte offsets of the 1D batch stage (strip_offset of
sf_batch_stage.h) against 64-bit arithmetic, at both ends of a row and on
both sides of column 2^29, where an offset from the row's start wraps."""
from tests import hostprog

PROGRAM = r"""
#include "sonic_amd.h"
#include "sf_batch_stage.h"
#include <cstdio>
using namespace sfamd;
int main() {
    for (long long n : {4LL, 70LL, (1LL << 29) - 3, (1LL << 29) + 64, (1LL << 30) + 5}) {
        GridDev G{};
        G.n[0] = (int)n;
        G.xo = 3;
        G.map_lo[0] = -1;
        G.map_hi[0] = (int)n;
        const int hi = (int)n - 2, last = hi + 3;
        for (int i0 : {0, 63, (hi / 63 - 1) * 63, hi / 63 * 63}) {
            if (i0 < 0 || i0 >= hi) continue;
            for (int t = 0; t < 64; ++t) {
                const int c = i0 + t < last ? i0 + t : last;
                const long long stored = c > n ? n : c;
                const long long want = (stored + 3) * 8, got = i0 * 8LL + strip_offset(G, i0, c);
                if (got != want) printf("n %lld i0 %d c %d: %lld, not %lld\n", n, i0, c, got, want);
            }
        }
    }
    printf("done\n");
}
"""


def test_offsets_of_long_rows(tmp_path):
    assert hostprog.run(tmp_path, PROGRAM) == ["done"]
