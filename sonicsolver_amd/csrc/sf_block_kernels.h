// sf_block_kernels.h -- the sweeps of small grids: a wave evaluates one face
// per lane and the waves of a block exchange the fluxes.
#pragma once

#include "sf_sweep_kernels.h"

namespace sfamd {

// ---------------------------------------------------------------------------
// A march evaluates the faces of its rows one after another, and on a grid of
// some 10^4 nodes that chain, two or three faces for one wave with a SIMD to
// itself, is what a stage takes.  Here every face of a block's rows has a
// wave of its own, and the waves exchange the fluxes through LDS: of
// `rows` rows, waves 0 .. rows take the y faces, waves rows + 1 .. 2 rows the
// upper x faces, and with 64 columns one more the first x faces.  The x waves
// then form the sums and the update, their operands requested before the
// Riemann solver.  Stencils are read from global memory, which the waves of a
// block share in the L1.  No march ring, so a wave takes 116 - 124 registers
// (WENO5, TENO5) and four run per SIMD.
//
// Faces, sums and updates are those of k_stage_yx, bit for bit.  The y faces
// at the ends of a block's rows are evaluated twice, so where the device is
// full the march is faster (yx_shape).  A pass of 20 steps with WENO5/HLLC:
// 40^2 0.67 -> 0.43 ms, 130^2 0.69 -> 0.45, 193 x 97 0.74 -> 0.58 (0.55 since
// the clock and the arguments cost less), 256^2 with TENO5/HLLC 1.12 -> 0.75
// (0.70), 400^2 1.24 -> 1.11.
// ---------------------------------------------------------------------------
constexpr int kBlockRows = 5;    // most rows of a block
constexpr int kBlockHalo7 = 4;   // ghost layers of WENO7

__host__ __device__ constexpr int block_waves(const YxShape& sh) {
    return 2 * sh.rows + 1 + (sh.cols == kXBlock);
}

template <int SCHEME>
struct BlockLds {
    double fy[kBlockRows + 1][5][kXBlock];
    double first[5][kBlockRows];
};

// Rows a0 .. a0 + rows - 1 (those up to the last advanced one) of plane k;
// lane t has column i0 + t.
template <int SCHEME, int FLUX, int TIME, bool HAS_S, bool CORNERS, int SLOTS, class Args>
__device__ __forceinline__ void block_yx_tile(const SweepArgs& W, const Args& args,
                                              BlockLds<SCHEME>& lds, int i0, int helper, int a0,
                                              int rows, int k, bool first_block) {
    constexpr int NS = Stencil<SCHEME>::ns;
    constexpr int H = NS / 2;
    const int t = threadIdx.x & (kXBlock - 1);
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kXBlock);
    const int i = i0 + t;
    const int hi0 = W.G.solved_hi[0];
    const int a1 = min(a0 + rows, W.G.solved_hi[1] + 1);
    const bool node = i <= hi0 && t >= helper;
    const int last = hi0 + H;
    unsigned flags = 0;
    double dt_local = INFINITY;
    // A fault was raised: keep the step-start state.  The waves of a block
    // may read it differently while another block raises it, so each drops
    // its own results only.
    const bool raised = *W.A.flags != 0;
    const StepClock clock(W.A);
    const double dt_lw = (FLUX == 5) ? clock.get(W.A) : 0.0;
    const double lwx = (FLUX == 5) ? dt_lw / W.G.d[0] : 0.0;   // Lax-Wendroff dt / spacing
    const double lwy = (FLUX == 5) ? dt_lw / W.G.d[1] : 0.0;
    const int xo = W.G.xo;
    const auto row_of = [&](const GridDev& G, int a) {
        return node_index(G, -xo, map_node(G, 1, a), k);
    };
    const unsigned own = (unsigned)(i + xo) * 8u;
    const unsigned off = (unsigned)(map_node(W.G, 0, min(i, last)) + xo) * 8u;
    const int a = a0 + w - rows - 1;   // an x wave's row
    const bool x_wave = w > rows && w <= 2 * rows && a < a1;
    double st[NS][5], f[5], ps[5], pq0[5];
    if (w <= rows) {
        const int ay = a0 + w;   // the face below row ay
        if (ay <= a1) {
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const long long row = row_of(W.G, ay - H + s);
#pragma unroll
                for (int v = 0; v < 5; ++v) st[s][v] = at(W.q + v * W.G.P + row, off);
            }
            unsigned fy = 0;
            face_flux<1, SCHEME, FLUX>(st, W.G.gamma, W.G.area[1], f, fy, lwy);
            if (!finite5(f)) fy |= kFlagFlux;
            if (node) flags |= fy;
#pragma unroll
            for (int v = 0; v < 5; ++v) lds.fy[w][v][t] = f[v];
        }
    } else if (w <= 2 * rows) {
        if (x_wave) {
            const long long row = row_of(W.G, a);
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const int c = map_node(W.G, 0, min(i - (H - 1) + s, last)) + xo;
#pragma unroll
                for (int v = 0; v < 5; ++v) st[s][v] = at(W.q + v * W.G.P + row, (unsigned)c * 8u);
            }
            unsigned fx = 0;
            face_flux_from<0, SCHEME, FLUX>(
                st,
                [&](int side, double (&b)[5]) {
                    if (side == 0) {
                        const SweepArgs& U = args();
#pragma unroll
                        for (int v = 0; v < 5; ++v) {
                            if (HAS_S) ps[v] = at(U.S + v * U.G.P + row, node ? own : off);
                            pq0[v] = at(U.A.q0 + v * U.G.P + row, node ? own : off);
                        }
                    }
#pragma unroll
                    for (int v = 0; v < 5; ++v) b[v] = st[H - 1 + side][v];
                },
                W.G.gamma, W.G.area[0], f, fx, lwx);
            if (!finite_sum5(f)) fx |= kFlagFlux;
            if (i <= hi0) flags |= fx;
        }
    } else if (a0 + t < a1) {
        // the first x faces (lower face of lane 0's node), lane r for row
        // a0 + r
        const long long row = row_of(W.G, a0 + t);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int c = map_node(W.G, 0, i0 - H + s) + xo;
#pragma unroll
            for (int v = 0; v < 5; ++v) st[s][v] = W.q[v * W.G.P + row + c];
        }
        face_flux<0, SCHEME, FLUX>(st, W.G.gamma, W.G.area[0], f, flags, lwx);
        if (!finite_sum5(f)) flags |= kFlagFlux;
#pragma unroll
        for (int v = 0; v < 5; ++v) lds.first[v][t] = f[v];
    }
    __syncthreads();
    const double dt_step = clock.get(W.A);
    if (first_block && w == 0) clock.commit(W.A, dt_step);
    if (raised) return;
    if (x_wave) {
        const int r = a - a0;
        double s5[5];
#pragma unroll
        for (int v = 0; v < 5; ++v) {
            const double up = lane_shift_up1(f[v]);
            const double lower = helper == 0 && t == 0 ? lds.first[v][r] : up;
            s5[v] = lds.fy[r + 1][v][t] - lds.fy[r][v][t];
            if (HAS_S) s5[v] = ps[v] + s5[v];
            s5[v] = s5[v] + (f[v] - lower);
        }
        if (node) {
            const SweepArgs& U = args();
            double dl = INFINITY, qn[5], pq[5];
            const long long nid = node_index(U.G, i, a, k);
#pragma unroll
            for (int v = 0; v < 5; ++v) pq[v] = st[H - 1][v];
            stage_update_dt<TIME>(U.G, U.A, nid, pq, pq0, s5, dt_step, flags, dl, qn);
            const SweepArgs& V = args();
            write_ends<CORNERS>(V.G, V.A.qout, i, a, k, nid, qn, flags);
            dt_local = dl;
        }
    }
    raise_fault(flags, W.A.flags, W.A.fault_tag, W.A.tag);
    if (W.A.reduce_dt && x_wave) wave_min_atomic<SLOTS>(dt_local, W.A.dtmin);
}

template <int SCHEME, int FLUX, int TIME, bool HAS_S>
__global__ __launch_bounds__(kXBlock * (2 * kBlockRows + 2)) void k_block_yx(SweepArgs W,
                                                                                  YxShape sh) {
    __shared__ BlockLds<SCHEME> lds;
    fetch_args<sizeof(SweepArgs)>();
    const unsigned chunk = gridDim.x >> 3;
    const unsigned bid = (blockIdx.x & 7u) * chunk + (blockIdx.x >> 3);
    if (bid >= sh.blocks) return;
    const unsigned bx = bid % (unsigned)sh.nx, br = bid / (unsigned)sh.nx;
    const int k = W.G.solved_lo[2] + (int)(br / (unsigned)sh.ny);
    const int a0 = W.G.solved_lo[1] + (int)(br % (unsigned)sh.ny) * sh.rows;
    const int helper = kXBlock - sh.cols;
    const int i0 = W.G.solved_lo[0] + (int)bx * sh.cols - helper;
    block_yx_tile<SCHEME, FLUX, TIME, HAS_S, false, kDtSlots>(
        W, [] () -> const SweepArgs& { return sweep_args(); }, lds, i0, helper, a0, sh.rows, k,
        bid == 0);
}

// z sweep of small grids (block_z_nodes): wave w of a block evaluates the
// face below the w-th node of its columns, and all but the last form their
// node's difference S from LDS.  Along x S is written without holes, as by
// k_sweep_march.
constexpr int kBlockZ = 7;

template <int SCHEME, int FLUX>
__global__ __launch_bounds__(kXBlock * (kBlockZ + 1)) void k_block_z(
    GridDev G, const double* __restrict__ q, double* __restrict__ S, StageArgs A) {
    constexpr int NS = Stencil<SCHEME>::ns;
    constexpr int H = NS / 2;
    __shared__ double fz[kBlockZ + 1][5][kXBlock];
    fetch_args<sizeof(GridDev) + 16 + sizeof(StageArgs)>();
    const bool raised = *A.flags != 0;   // as in block_yx_tile
    const int t = threadIdx.x & (kXBlock - 1);
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kXBlock);
    const int seg = blockDim.x / kXBlock - 1;
    const int i = blockIdx.x * kXBlock + t;
    const int ic = min(max(i, G.solved_lo[0]), G.solved_hi[0]);
    const int j = G.solved_lo[1] + blockIdx.y;
    const int a = G.solved_lo[2] + blockIdx.z * seg + w;   // the face below node a
    const double lw = (FLUX == 5) ? StepClock(A).get(A) / G.d[2] : 0.0;
    unsigned flags = 0;
    if (a <= G.solved_hi[2] + 1) {
        double st[NS][5], f[5];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const long long id = node_index(G, ic, j, map_node(G, 2, a - H + s));
#pragma unroll
            for (int v = 0; v < 5; ++v) st[s][v] = q[v * G.P + id];
        }
        face_flux<2, SCHEME, FLUX>(st, G.gamma, G.area[2], f, flags, lw);
#pragma unroll
        for (int v = 0; v < 5; ++v) {
            if (!isfinite(f[v])) flags |= kFlagFlux;
            fz[w][v][t] = f[v];
        }
    }
    __syncthreads();
    if (raised) return;
    if (w < seg && a <= G.solved_hi[2] && i < G.n[0]) {
        const long long id = node_index(G, i, j, a);
#pragma unroll
        for (int v = 0; v < 5; ++v) S[v * G.P + id] = fz[w + 1][v][t] - fz[w][v][t];
    }
    raise_fault(flags, A.flags, A.fault_tag, A.tag);
}

}  // namespace sfamd
