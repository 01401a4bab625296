// sf_batch_stage.h -- the stage kernels of batched problems: one RK stage of
// every live problem, over a table of tiles.
#pragma once

#include "sf_sweep_kernels.h"

namespace sfamd {

// Partial minima of a problem's CFL accumulator (kDtStride apart).  Its
// blocks number at most a few hundred, so fewer than a grid's 64 do.
constexpr int kItemDtSlots = 8;

// Arguments of a problem's three SSPRK3 stages, in device memory.
struct ItemArgs {
    SweepArgs stage[3];
};

// One tile of a problem, the work of a wave.  Of a 2D problem: rows a0 ..
// a1-1, lane t in column i0 + t, where lane 0 only evaluates a face if
// helper is set.  Of a 1D one: `a0` strips of 63 nodes, the first strip's
// lane 0 in column i0.
struct BatchTile {
    int slot;
    int i0;
    int a0;
    int a1;   // with helper in bit 31
};

// A problem's arguments as the tile reads them: like sweep_args(), what is
// read through it is loaded where it is used, by scalar loads from the
// constant cache, instead of held in scalar registers.
struct ItemArgsAt {
    const SweepArgs* at;
    __device__ __forceinline__ const SweepArgs& operator()() const {
        auto p = (const __attribute__((address_space(4))) SweepArgs*)at;
        asm volatile("" : "+s"(p));
        return *(const SweepArgs*)p;
    }
};

struct BatchStage {
    const ItemArgs* items;
    const int* live;          // by slot: the problem takes this step
    const BatchTile* tiles;
    int stage;
};

__device__ __forceinline__ const BatchTile batch_tile(const BatchStage& B, int tile) {
    const BatchTile T = B.tiles[tile];
    BatchTile u;
    u.slot = __builtin_amdgcn_readfirstlane(T.slot);
    u.i0 = __builtin_amdgcn_readfirstlane(T.i0);
    u.a0 = __builtin_amdgcn_readfirstlane(T.a0);
    u.a1 = __builtin_amdgcn_readfirstlane(T.a1);
    return u;
}

// The stage of 2D problems: y and x faces and the update of a tile at once,
// ends written in place, as on a grid (k_stage_yx).  The waves are bound by
// FP64 issue where they fill the device, by their serial chain of faces
// where they do not; the tile's rows are chosen by the cost of both over the
// whole batch.  Separate y and x sweeps with S between them, 64 x 32 tiles
// and four ghost fills per stage took, per step with WENO5/HLLC, 273 us for
// one problem of 131^2, 1318 for 200 and 1079 for 12 of 512^2; this takes
// 40, 817 and 569.
template <int SCHEME, int FLUX>
__device__ __forceinline__ void plane_tiles(const BatchStage& B, YxLds<SCHEME>& lds, int t0,
                                            int t1, int b0, int nb) {
#pragma clang loop unroll(disable)
    for (int tile = t0 + b0; tile < t1; tile += nb) {
        const BatchTile T = batch_tile(B, tile);
        if (!B.live[T.slot]) continue;   // fixed during a step
        const ItemArgsAt args{&B.items[T.slot].stage[B.stage]};
        wave_lds_order();   // after the tile before
        stage_yx_tile<SCHEME, FLUX, SF_TIME_SSPRK3, false, true, kItemDtSlots, 1>(
            args(), args, lds, T.i0, (int)((unsigned)T.a1 >> 31), T.a0, T.a1 & 0x7fffffff, 0,
            false, 0u);
    }
}

// Byte offset, from column i0 of the row at `xo`, of the stored node that
// stands for column c >= i0 of a strip that starts there.  From the row's
// start it would pass 2^32 at column 2^29, and an arena holds longer
// problems.
__host__ __device__ __forceinline__ unsigned strip_offset(const GridDev& G, int i0, int c) {
    return (unsigned)(map_node(G, 0, c) - i0 + G.xo) * 8u;
}

// The stage of 1D problems: a wave takes strips of 63 nodes, lane 0
// evaluating the first one's lower face.  Bound like the planes' tiles: 300
// problems of 8192 nodes take 271 us per step, 2.2 us of issue per strip and
// SIMD (390 in multi-wave tiles with two fills per stage), 16 of 300 nodes
// 27 us (41).
template <int SCHEME, int FLUX>
__device__ __forceinline__ void line_tiles(const BatchStage& B, double (&row)[5][kXBlock + 6],
                                           int t0, int t1, int b0, int nb) {
    constexpr int H = 3;
    static_assert(Stencil<SCHEME>::ns == 2 * H, "a six-node stencil");
    const int t = threadIdx.x;
    // halo: lane l < 25 loads variable l / 5, halo column l % 5
    const int hv = t / (2 * H - 1), hc = t % (2 * H - 1);
    const bool halo = hv < 5;
    const int hcol = hc < H - 1 ? hc - (H - 1) : kXBlock + hc - (H - 1);   // from i0
#pragma clang loop unroll(disable)
    for (int tile = t0 + b0; tile < t1; tile += nb) {
        const BatchTile T = batch_tile(B, tile);
        if (!B.live[T.slot]) continue;   // fixed during a step
        const ItemArgsAt args{&B.items[T.slot].stage[B.stage]};
        const SweepArgs& W = args();
        const double dt_step = *W.A.dt;
        const int hi0 = W.G.solved_hi[0];
        const int last = hi0 + H;   // the last column a face reads
        unsigned flags = 0;
        double dt_local = INFINITY;
        int i0 = T.i0;
#pragma clang loop unroll(disable)
        for (int s = 0; s < T.a0 && i0 < hi0; ++s, i0 += kXBlock - 1) {
            const SweepArgs& U = args();
            const int i = i0 + t;
            const bool node = i <= hi0 && t >= 1;
            const unsigned off = strip_offset(U.G, i0, min(i, last));
            double pq[5], pq0[5];
#pragma unroll
            for (int v = 0; v < 5; ++v) pq[v] = at(U.q + v * U.G.P + i0, off);
            double h = 0.0;
            if (halo) h = U.q[hv * U.G.P + (map_node(U.G, 0, min(i0 + hcol, last)) + U.G.xo)];
            wave_lds_order();
#pragma unroll
            for (int v = 0; v < 5; ++v) row[v][t + H - 1] = pq[v];
            if (halo) row[hv][hcol + H - 1] = h;
            wave_lds_order();
            double st[2 * H][5];
#pragma unroll
            for (int x = 0; x < 2 * H; ++x)
#pragma unroll
                for (int v = 0; v < 5; ++v) st[x][v] = row[v][t + x];
            unsigned fx = 0;
            double f5[5];
            face_flux_from<0, SCHEME, FLUX>(
                st,
                [&](int side, double (&b)[5]) {
                    if (side == 0) {
                        const SweepArgs& V = args();
#pragma unroll
                        for (int v = 0; v < 5; ++v) pq0[v] = at(V.A.q0 + v * V.G.P + i0, off);
                    }
#pragma unroll
                    for (int v = 0; v < 5; ++v) b[v] = row[v][t + H - 1 + side];
                },
                U.G.gamma, U.G.area[0], f5, fx, 0.0);
            if (!finite_sum5(f5)) fx |= kFlagFlux;
            if (i <= hi0) flags |= fx;
            double s5[5];
#pragma unroll
            for (int v = 0; v < 5; ++v) s5[v] = f5[v] - lane_shift_up1(f5[v]);
            if (node) {
                const SweepArgs& V = args();
#pragma unroll
                for (int v = 0; v < 5; ++v) pq[v] = row[v][t + H - 1];
                double dl = INFINITY, qn[5];
                const long long id = i + V.G.xo;
                stage_update_dt<SF_TIME_SSPRK3>(V.G, V.A, id, pq, pq0, s5, dt_step, flags, dl, qn);
                const SweepArgs& X = args();
                write_ends<false, false>(X.G, X.A.qout, i, 0, 0, id, qn, flags);
                dt_local = fmin(dt_local, dl);
            }
        }
        const SweepArgs& Z = args();
        raise_fault(flags, Z.A.flags, Z.A.fault_tag, Z.A.tag);
        if (Z.A.reduce_dt) wave_min_atomic<kItemDtSlots>(dt_local, Z.A.dtmin);
    }
}

// Tile ranges and block ranges of the four (scheme, flux) variants,
// variant v = 2*scheme + flux.
struct Split {
    int tile[5];
    int block[5];
};

// The LDS of whichever variant a block runs.
union PlaneLds {
    __device__ PlaneLds() {}
    YxLds<0> weno5;
    YxLds<1> teno5;
};

// Every variant present in one launch: block ranges are assigned to variants.
template <bool PLANE>
__global__ __launch_bounds__(kXBlock)
__attribute__((amdgpu_waves_per_eu(3, 8))) void k_batch_stage_mixed(BatchStage B, Split sp) {
    __shared__ PlaneLds lds;
    __shared__ double row[5][kXBlock + 6];
    const int bid = blockIdx.x;
    int v = 0;
    while (v < 3 && bid >= sp.block[v + 1]) ++v;
    const int t0 = sp.tile[v], t1 = sp.tile[v + 1];
    const int b0 = bid - sp.block[v], nb = sp.block[v + 1] - sp.block[v];
    if (PLANE) {
        switch (v) {
        case 0: plane_tiles<0, 0>(B, lds.weno5, t0, t1, b0, nb); break;
        case 1: plane_tiles<0, 1>(B, lds.weno5, t0, t1, b0, nb); break;
        case 2: plane_tiles<1, 0>(B, lds.teno5, t0, t1, b0, nb); break;
        default: plane_tiles<1, 1>(B, lds.teno5, t0, t1, b0, nb); break;
        }
    } else {
        switch (v) {
        case 0: line_tiles<0, 0>(B, row, t0, t1, b0, nb); break;
        case 1: line_tiles<0, 1>(B, row, t0, t1, b0, nb); break;
        case 2: line_tiles<1, 0>(B, row, t0, t1, b0, nb); break;
        default: line_tiles<1, 1>(B, row, t0, t1, b0, nb); break;
        }
    }
}

// One variant per launch.
template <bool PLANE, int SCHEME, int FLUX>
__global__ __launch_bounds__(kXBlock)
__attribute__((amdgpu_waves_per_eu(3, 8))) void k_batch_stage(BatchStage B, int t0, int t1) {
    if constexpr (PLANE) {
        __shared__ YxLds<SCHEME> lds;
        plane_tiles<SCHEME, FLUX>(B, lds, t0, t1, blockIdx.x, gridDim.x);
    } else {
        __shared__ double row[5][kXBlock + 6];
        line_tiles<SCHEME, FLUX>(B, row, t0, t1, blockIdx.x, gridDim.x);
    }
}

}  // namespace sfamd
