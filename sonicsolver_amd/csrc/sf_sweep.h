// sf_sweep.h -- launch of one sweep (one axis of one stage) of the grid
// path.  Each reconstruction scheme's kernels are compiled in a translation
// unit of their own (sf_sweep_<scheme>.hip instantiates launch_sweep for
// its scheme id), so the twenty scheme x flux combinations build in
// parallel.
#pragma once

#include "sf_block_kernels.h"

#include <algorithm>

namespace sfamd {

struct SweepCall {
    GridDev G;
    const double* q;   // stage input state (ghosts filled)
    double* S;         // flux-difference accumulator
    StageArgs A;
    hipStream_t stream;
    int seg;           // base nodes per march segment (y and z sweeps)
    int cus;           // compute units of the device
    int x_walk;        // x sweep by lines (1), by flat tiles (0), automatic (-1)
};

// Cost, in face evaluations of one wave, of a march whose one-wave blocks
// evaluate `faces` faces each, on a device of `cus` compute units (four SIMDs
// each).  Blocks are dealt evenly, so the SIMD with the most of them sets the
// time.  Measured on 2D and 3D grids with the fused y / x march: one wave on
// a SIMD takes 1.73 times as long per face as each of three or more, two
// take 1.3 times, and a block's start (its window's loads) costs as much as
// five faces where nothing hides it and 1.5 where other waves do.
// 853^2, WENO5/HLLC, per stage: 52 us with 1008 blocks of 12 rows, 73 with
// 1092 of 11, 47 with 2002 of 6, 45 with 2996 of 4.
inline double march_cost(long long blocks, double faces, int cus) {
    const long long simds = 4LL * std::max(cus, 8);
    const long long w = (blocks + simds - 1) / simds;
    if (w <= 1) return 1.73 * (faces + 5.0);
    if (w == 2) return 2.6 * (faces + 4.0);
    return 1.07 * (double)w * (faces + (w <= 4 ? 3.0 : 1.5));
}

// Waves on the busiest SIMD when `blocks` blocks of `waves` waves are dealt
// evenly to the compute units.
inline long long waves_per_simd(long long blocks, int waves, int cus) {
    const long long units = std::max(cus, 8);
    return (blocks + units - 1) / units * ((waves + 3) / 4);
}

inline long long block_load(const YxShape& sh, int cus) {
    return waves_per_simd(sh.blocks, block_waves(sh), cus);
}

// Nodes along z of a block of the z sweep of small grids (k_block_z), whose
// blocks take `columns` columns of 64 nodes, or 0 where the march takes it:
// where the device does not hold all blocks at once.  With WENO5/HLLC a pass
// of 20 steps on 24^3 takes 0.96 ms by the march and 0.86 by blocks, on 48^3
// 1.75 and 1.50 (three waves per SIMD), on 100 x 40 x 40 2.02 and 1.92 (four);
// on 64^3, with six, 2.56 and 3.16.
template <int SCHEME>
int block_z_nodes(long long columns, int nz, int cus) {
    int best = 0;
    long long least = SCHEME == 3 ? 3 : 5;
    for (int nodes : {7, 3}) {
        const long long w = waves_per_simd(columns * ((nz + nodes - 1) / nodes), nodes + 1, cus);
        if (w >= least) continue;
        least = w;
        best = nodes;
    }
    return best;
}

// Grid of the x sweep (a multiple of 8 for the XCD mapping): one block per
// 128 tiles, at least as many as the device holds at once (compute units x
// the kernel's resident blocks per unit) and at most 16384.  Blocks beyond
// the resident ones run in rounds, each paying its start-up again, which
// costs most where a block gets few tiles: the 2048^2 x sweep ran 0.46 ms
// with 16384 blocks (4 tiles each) and 0.32 ms with one resident round;
// 256^3 1.07 and 0.78 ms.  Long runs per block balance worse: 512^3 ran
// 6.06 ms with 16384 blocks (130 tiles each) and 6.19 ms with one round.
template <int SCHEME, int FLUX, int TIME>
unsigned x_blocks(int cus, long long tiles) {
    static int per_cu = 0;   // one per kernel instantiation
    if (per_cu == 0) {
        int n = 0;
        per_cu = (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                      &n, k_sweep_x<SCHEME, FLUX, TIME>, kXBlock, 0) == hipSuccess && n > 0)
                     ? n : 8;
    }
    const long long resident = (long long)std::max(cus, 8) * per_cu;
    const long long want = std::min<long long>(std::max<long long>(tiles / 128, resident), 16384);
    return (unsigned)((std::min<long long>(tiles, want) + 7) & ~7LL);
}

// The x sweep is always the last sweep of a stage (x is always active and
// the sweeps run z, y, x), so it is compiled in its final mode only, and the
// y / z marches in their S-writing modes only.  Returns -1 for a combination
// that is not compiled.
template <int SCHEME, int FLUX, int MODE>
int launch_sweep_fm(const SweepCall& c, int axis) {
    const GridDev& G = c.G;
    if (axis == 0) {
        if constexpr (MODE != kFinal) {
            return -1;
        } else {
            // What comes here (yx_shape): residuals, 1D grids, 2D and 3D ones
            // narrower than 32 nodes that fill the device, and a chosen walk.
            // Grids of 64 columns and at least 256 x lines per CU (16 for
            // every wave slot at four waves per SIMD) walk whole lines, which
            // by itself only residuals of large grids do: their x sweep on
            // 256^3 takes 0.49 ms against 0.53 with the flattened tiles with
            // WENO5/HLLC, 0.74 against 0.81 with TENO5, 0.78 against 0.85 with
            // WENO7, 0.47 against 0.51 with WENO3, on 384^3 2.30 against 2.43;
            // with too few lines to fill the device, on 128^3, 0.078 against
            // 0.074.
            // The line walk addresses a lane's stage operands by a 32-bit
            // byte offset of up to one variable (8 P bytes) past the tile.
            const SweepArgs W{G, c.q, c.S, c.A};
            const long long lines = (long long)G.n[1] * G.n[2];
            const bool fits = (long long)G.P * 8 + 1024 < (1LL << 32);
            const bool by_lines =
                fits && (c.x_walk == 1 ||
                         (c.x_walk < 0 && G.n[0] >= kXBlock &&
                          lines >= 256LL * std::max(c.cus, 8)));
            if (by_lines) {
                const long long groups = (lines + kLineGroup - 1) / kLineGroup;
                const unsigned nb = (unsigned)std::min<long long>(groups, 16384);
#define SF_LAUNCH_XL(T) \
    k_sweep_xl<SCHEME, FLUX, T><<<nb, kXBlock, 0, c.stream>>>(W)
                switch (c.A.time) {
                case 0: SF_LAUNCH_XL(0); break;
                case 1: SF_LAUNCH_XL(1); break;
                case 2: SF_LAUNCH_XL(2); break;
                default: SF_LAUNCH_XL(3); break;
                }
#undef SF_LAUNCH_XL
                return 0;
            }
            // one resident block per slot, each looping over tiles of
            // kXBlock faces
            const long long faces = (long long)(G.n[0] + 1) * G.n[1] * G.n[2];
            const long long tiles = (faces - 1 + kXBlock - 2) / (kXBlock - 1);
#define SF_LAUNCH_X(T)                                                            \
    k_sweep_x<SCHEME, FLUX, T><<<x_blocks<SCHEME, FLUX, T>(c.cus, tiles), kXBlock, 0, \
                                c.stream>>>(W)
            switch (c.A.time) {
            case 0: SF_LAUNCH_X(0); break;
            case 1: SF_LAUNCH_X(1); break;
            case 2: SF_LAUNCH_X(2); break;
            default: SF_LAUNCH_X(3); break;
            }
#undef SF_LAUNCH_X
            return 0;
        }
    }
    if constexpr (MODE == kFinal) {
        return -1;
    } else {
        // the advanced nodes along each axis
        const auto span = [&](int a) { return G.solved_hi[a] - G.solved_lo[a] + 1; };
        const unsigned other = (unsigned)span(3 - axis);
        const unsigned cols = (unsigned)((G.n[0] + kMarchBlock - 1) / kMarchBlock);
        // Each segment re-reads the stencil window and evaluates one extra
        // face at its start; march_cost weighs that against filling the
        // chip.  A face's arithmetic does not depend on the segment length,
        // so neither does the result.  c.seg > 0 fixes the length instead.
        int seg = c.seg;
        if constexpr (MODE == kCopyS) {
            const int nodes = axis == 2 && seg <= 0
                                  ? block_z_nodes<SCHEME>((long long)cols * other, span(2), c.cus)
                                  : 0;
            if (nodes > 0) {
                const dim3 grid(cols, other, (unsigned)((span(2) + nodes - 1) / nodes));
                k_block_z<SCHEME, FLUX><<<grid, kXBlock * (nodes + 1), 0, c.stream>>>(G, c.q, c.S,
                                                                                      c.A);
                return 0;
            }
        }
        if (seg <= 0) {
            double least = 0.0;
            for (int s = 1; s <= 64; ++s) {
                const long long blocks = (long long)cols * other * ((span(axis) + s - 1) / s);
                const double cost = march_cost(blocks, s + 1.0, c.cus);
                if (seg > 0 && cost >= least) continue;
                least = cost;
                seg = s;
            }
        }
        const dim3 grid(cols, other, (unsigned)((span(axis) + seg - 1) / seg));
        if (axis == 1)
            k_sweep_march<1, SCHEME, FLUX, MODE><<<grid, kMarchBlock, 0, c.stream>>>(
                G, c.q, c.S, c.A, seg);
        else
            k_sweep_march<2, SCHEME, FLUX, MODE><<<grid, kMarchBlock, 0, c.stream>>>(
                G, c.q, c.S, c.A, seg);
        return 0;
    }
}

template <int SCHEME, int FLUX>
int launch_sweep_f(const SweepCall& c, int axis, int mode) {
    if (mode == kCopyS) return launch_sweep_fm<SCHEME, FLUX, kCopyS>(c, axis);
    if (mode == kAccumS) return launch_sweep_fm<SCHEME, FLUX, kAccumS>(c, axis);
    return launch_sweep_fm<SCHEME, FLUX, kFinal>(c, axis);
}

// The y and x faces and the stage update in one launch (k_stage_yx).
// Returns -1 for a time recipe that is not compiled.
template <int SCHEME, int FLUX>
int launch_yx_f(const SweepCall& c, const YxShape& sh) {
    const SweepArgs W{c.G, c.q, c.S, c.A};
    const unsigned nb = (sh.blocks + 7) & ~7u;
    const unsigned wg = kXBlock * block_waves(sh);
#define SF_LAUNCH_YX(T)                                                                       \
    do {                                                                                      \
        if (sh.block && c.G.active[2])                                                        \
            k_block_yx<SCHEME, FLUX, T, true><<<nb, wg, 0, c.stream>>>(W, sh);                \
        else if (sh.block)                                                                    \
            k_block_yx<SCHEME, FLUX, T, false><<<nb, wg, 0, c.stream>>>(W, sh);               \
        else if (sh.waves > 1 && c.G.active[2])                                               \
            k_stage_yx<SCHEME, FLUX, T, true, kYxWaves>                                       \
                <<<nb, kXBlock * kYxWaves, 0, c.stream>>>(W, sh);                             \
        else if (sh.waves > 1)                                                                \
            k_stage_yx<SCHEME, FLUX, T, false, kYxWaves>                                      \
                <<<nb, kXBlock * kYxWaves, 0, c.stream>>>(W, sh);                             \
        else if (c.G.active[2])                                                               \
            k_stage_yx<SCHEME, FLUX, T, true, 1><<<nb, kXBlock, 0, c.stream>>>(W, sh);        \
        else                                                                                  \
            k_stage_yx<SCHEME, FLUX, T, false, 1><<<nb, kXBlock, 0, c.stream>>>(W, sh);       \
    } while (0)
    switch (c.A.time) {
    case 0: SF_LAUNCH_YX(0); break;
    case 1: SF_LAUNCH_YX(1); break;
    case 2: SF_LAUNCH_YX(2); break;
    default: return -1;
    }
#undef SF_LAUNCH_YX
    return 0;
}

template <int SCHEME>
int launch_yx(const SweepCall& c, int flux, const YxShape& sh) {
    switch (flux) {
    case 0: return launch_yx_f<SCHEME, 0>(c, sh);
    case 1: return launch_yx_f<SCHEME, 1>(c, sh);
    case 2: return launch_yx_f<SCHEME, 2>(c, sh);
    case 3: return launch_yx_f<SCHEME, 3>(c, sh);
    case 4: return launch_yx_f<SCHEME, 4>(c, sh);
    default: return launch_yx_f<SCHEME, 5>(c, sh);
    }
}

// One sweep of scheme SCHEME with face flux `flux` (SF_FLUX_*) along
// `axis` in stage mode `mode` (kCopyS, kAccumS, kFinal).
template <int SCHEME>
int launch_sweep(const SweepCall& c, int flux, int axis, int mode) {
    switch (flux) {
    case 0: return launch_sweep_f<SCHEME, 0>(c, axis, mode);
    case 1: return launch_sweep_f<SCHEME, 1>(c, axis, mode);
    case 2: return launch_sweep_f<SCHEME, 2>(c, axis, mode);
    case 3: return launch_sweep_f<SCHEME, 3>(c, axis, mode);
    case 4: return launch_sweep_f<SCHEME, 4>(c, axis, mode);
    default: return launch_sweep_f<SCHEME, 5>(c, axis, mode);
    }
}

extern template int launch_sweep<0>(const SweepCall&, int, int, int);
extern template int launch_sweep<1>(const SweepCall&, int, int, int);
extern template int launch_sweep<2>(const SweepCall&, int, int, int);
extern template int launch_sweep<3>(const SweepCall&, int, int, int);
extern template int launch_yx<0>(const SweepCall&, int, const YxShape&);
extern template int launch_yx<1>(const SweepCall&, int, const YxShape&);
extern template int launch_yx<2>(const SweepCall&, int, const YxShape&);
extern template int launch_yx<3>(const SweepCall&, int, const YxShape&);

// Shape of a launch of k_block_yx over nx x ny x nz advanced nodes: the rows
// and columns of a block with the least load.  A block's 2 rows + 1 waves,
// one more with 64 columns, fill the four SIMDs evenly, or all but one wave,
// with an odd number of rows.
inline YxShape block_shape(int nx, int ny, int nz, int cus) {
    YxShape best{};
    for (int cols = kXBlock - 1; cols <= kXBlock; ++cols)
        for (int rows = 1; rows <= kBlockRows; rows += 2) {
            YxShape sh{};
            sh.cols = cols;
            sh.rows = rows;
            sh.nx = (nx + cols - 1) / cols;
            sh.ny = (ny + rows - 1) / rows;
            const long long blocks = (long long)sh.nx * sh.ny * nz;
            if (blocks > 1LL << 24) continue;
            sh.blocks = (unsigned)blocks;
            sh.block = 1;
            if (!best.blocks || block_load(sh, cus) < block_load(best, cus)) best = sh;
        }
    return best;
}

// Shape of the fused y / x launch of a stage, or blocks = 0 where the
// separate sweeps take it: the residual-only mode, a chosen x walk, and grids
// narrower than half a wave that fill the device more than twice over, whose
// x faces the flattened tiles pack into whole waves (24 x 200 x 200,
// WENO5/HLLC, 3 steps: 2.64 ms separately, 2.73 fused; 32 x 150 x 150: 1.91
// and 1.93; 40 x 100 x 100: 1.41 and 1.30).  Everywhere else the fused
// launch was faster, e.g. 512^3 77.3 -> 72.0 ms a pass of two steps, 2048^2
// TENO5/HLLC 6.39 -> 5.75, 853^2 5.22 -> 4.23, 256^2 TENO5/HLLC 2.40 ->
// 1.36, 64^3 4.32 -> 2.87, 40^2 1.05 -> 0.76 (the small ones by shorter
// segments in the z march, too).
//
// Blocks of four waves: 853^2 2.94 -> 2.83 ms a pass of 20 steps, 600^2 1.82
// -> 1.71, 64^3 2.49 -> 2.38, 1000^2 (10 steps) 2.03 -> 1.94, 900^2 with
// TENO5/HLLC 2.45 -> 2.37; with the long tiles of the largest grids there is
// little to share, and they take one (512^3 71.6 ms, 72.9 with four; on
// 2048^2 with TENO5/HLLC four waves of eight rows take 5.06 against the 5.13
// of the long single ones, which the cost does not see).
//
// Small grids take k_block_yx, up to the number of waves per SIMD at which it
// stays ahead of the march with every scheme: 8 in 2D (400^2, passes of 20
// steps: WENO5/HLLC 1.11 ms against 1.24, TENO5/HLLC 1.38 against 1.59,
// WENO3/HLLC 0.86 against 0.98; at 12, 500^2, 1.50 against 1.45, 1.90 against
// 1.80 and 1.13 against 1.11), 6 in 3D (48^3 with WENO5/HLLC 1.75 against
// 1.90; at 8, 100 x 40 x 40, 2.16 against 2.02) and 4 with WENO7, of which
// three waves fit a SIMD (10 RK4 steps on 300^2 0.71 against 0.83; at 8,
// 400^2, 1.18 against 1.14).
inline YxShape yx_shape(const SweepCall& c) {
    YxShape best{};
    const GridDev& G = c.G;
    if (!G.active[1] || c.x_walk >= 0 || c.A.time == 3) return best;
    const int nx = G.solved_hi[0] - G.solved_lo[0] + 1, ny = G.solved_hi[1] - G.solved_lo[1] + 1;
    const int nz = G.solved_hi[2] - G.solved_lo[2] + 1;
    if (c.seg <= 0) {
        const YxShape sh = block_shape(nx, ny, nz, c.cus);
        const long long most = G.g[0] == kBlockHalo7 ? 4 : G.active[2] ? 6 : 8;
        if (block_load(sh, c.cus) <= most) return sh;
    }
    double least = 0.0;
    // columns a block advances: 64 with its first x faces evaluated
    // beforehand, or 63 with lane 0 evaluating them; one wave per block, whose
    // rows' first y face the block below evaluates, too, or kYxWaves, which
    // share theirs
    for (int waves = 1; waves <= kYxWaves; waves += kYxWaves - 1)
        for (int cols = kXBlock; cols >= kXBlock - 1; --cols) {
            YxShape sh{};
            sh.cols = cols;
            sh.waves = waves;
            sh.nx = (nx + cols - 1) / cols;
            const int most = waves > 1 && cols == kXBlock ? kYxWaveRows : kYxRows;
            for (int rows = 1; rows <= most; ++rows) {
                if (c.seg > 0 && (waves > 1 || rows != std::min(c.seg, kYxRows))) continue;
                sh.rows = rows;
                sh.ny = (ny + rows * waves - 1) / (rows * waves);
                const long long blocks = (long long)sh.nx * sh.ny * nz;
                const double faces = 2.0 * rows + 1.0 / waves + (cols == kXBlock ? 1.0 : 0.0);
                const double cost = march_cost(blocks * waves, faces, c.cus);
                if (best.blocks && cost >= least) continue;
                least = cost;
                best = sh;
                best.blocks = (unsigned)blocks;
            }
        }
    if (2 * G.n[0] < kXBlock &&
        (long long)best.blocks * best.waves > 8LL * std::max(c.cus, 8))
        best.blocks = 0;
    return best;
}

}  // namespace sfamd
