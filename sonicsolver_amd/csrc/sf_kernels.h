// sf_kernels.h -- gfx950 kernels of the explicit Euler hot path besides the
// sweeps (included by sf_capi.hip; the sweeps are in sf_sweep_kernels.h).
//
// Data layout in HBM: conserved state as structure-of-arrays FP64,
// q[v*P + (k*m1 + j)*m0 + i], with a ghost layer as deep as the scheme's
// halo (2 for WENO3, 3 for WENO5 / TENO5, 4 for WENO7) on every active axis
// (m_d = n_d + 2 g) and none on an inactive one.  Work per RK stage:
//
//   boundary closure             none of its own: k_stage_yx writes the
//                                boundary node and the first ghost next to a
//                                node it advances at a zeroGradient end, and
//                                the marches read the node that stands for a
//                                ghost (map_node); k_fill stores all ghosts
//                                after an upload and for the separate x sweeps
//   z sweep                      k_sweep_march: one lane per (x, column
//                                               segment), marching along the
//                                               axis with the stencil window
//                                               in LDS, so each node is
//                                               loaded once and each face
//                                               evaluated once
//   y and x sweeps               k_stage_yx:    the same march along y with
//                                               the x faces of each row taken
//                                               from the window's rows
//   both on small grids          k_block_z, k_block_yx: a wave per face
//   separately, where yx_shape   k_sweep_march, then k_sweep_x (one lane per
//   says so                      x face, the flux difference by a cross-lane
//                                shift) or k_sweep_xl (whole lines in 64-node
//                                tiles)
//   the last launch also applies the stage update, validates the new state
//   and (on the last stage) folds the CFL scan of the next step into a
//   wave-level minimum (DPP moves) plus one 64-bit atomic per wave.
//
// Sweeps accumulate S = sum_d (F_d(i) - F_d(i-1)) and the update multiplies
// by Jac once, as Math::localSpatialResidual does
// (SF_residualAssembly.h:12-32).
#pragma once

#include "sf_step1d.h"
#include "sf_sweep_kernels.h"

namespace sfamd {

// ---------------------------------------------------------------------------
// Standalone CFL scan (first step, or sf_compute_dt).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_cfl(GridDev G, const double* __restrict__ q, double cfl,
                                             unsigned long long* slots, Fault* fault,
                                             long long tag) {
    if (fault->flags) return;
    const unsigned N = (unsigned)G.n[0] * G.n[1] * G.n[2];   // at most 2^31
    unsigned flags = 0;
    double best = INFINITY;
    for (unsigned long long u = blockIdx.x * blockDim.x + threadIdx.x; u < N;
         u += gridDim.x * blockDim.x) {
        const unsigned line = (unsigned)u / (unsigned)G.n[0];
        const int i = (int)((unsigned)u - line * (unsigned)G.n[0]);
        const unsigned kz = fast_div(line, G.div_n1);
        const int j = (int)(line - kz * (unsigned)G.n[1]), k = (int)kz;
        if (!solved_node(G, i, j, k)) continue;
        const long long id = node_index(G, i, j, k);
        double qq[5];
#pragma unroll
        for (int v = 0; v < 5; ++v) qq[v] = q[v * G.P + id];
        best = fmin(best, local_dt(G, qq, cfl, flags));
    }
    raise_fault(flags, &fault->flags, &fault->tag, tag);
    wave_min_atomic(best, slots);
}

// The clock between two steps, by one wave: commit the step just taken, then
// form the next step's dt from the CFL accumulator, which is reset for the
// scan after it.  Nothing once a fault is raised.  snap (host memory, may be
// null) receives the clock and the fault record as they are afterwards.
__global__ __launch_bounds__(kDtSlots) void k_clock(Control* c, unsigned long long* slots,
                                                    double* dt_hist, int slot, int commit,
                                                    int next_dt, Control* snap) {
    const int t = threadIdx.x;
    if (t == 0) c->fault.before = c->fault.flags;
    if (!c->fault.flags) {
        if (commit && t == 0) {
            c->clock.time += c->clock.dt;
            c->clock.steps += 1;
        }
        if (next_dt) {
            const unsigned long long b = wave_min_bits(slots[t * kDtStride]);
            slots[t * kDtStride] = 0x7FF0000000000000ull;
            if (t == 0) {
                double dt = __longlong_as_double((long long)b);
                dt = fmin(dt, c->clock.max_dt);
                dt = fmin(dt, c->clock.limit);
                c->clock.dt = dt;
                if (dt_hist) dt_hist[slot] = dt;
            }
        }
    }
    if (snap && t == 0) *snap = *c;
}

// After the last step of a run whose steps keep the clock: commit it, hand the CFL scan it folded to
// the grid's accumulator and clear the three that the steps used in turn.
__global__ __launch_bounds__(kDtSlots) void k_close_run(Control* c, unsigned long long* slots,
                                                       const unsigned long long* scan,
                                                       unsigned long long* sets, Control* snap) {
    const int t = threadIdx.x;
    if (!c->fault.flags) {
        if (t == 0) {
            c->clock.time += c->clock.dt;
            c->clock.steps += 1;
        }
        slots[t * kDtStride] = scan[t * kDtStride];
    } else if (t == 0 && c->fault.stages) {
        // tiles run their stages independently: the record is the earliest
        // stage's, whose flags a launch per stage would have stopped at
        const int s = (__ffs((int)c->fault.stages) - 1) / 8;
        c->fault.flags = (c->fault.stages >> (8 * s)) & 0xffu;
        c->fault.stages = 0u;
    }
    for (int s = 0; s < kStepSets; ++s)
        sets[(s * kDtSlots + t) * kDtStride] = 0x7FF0000000000000ull;
    if (snap && t == 0) *snap = *c;
}

__global__ void k_set_dt(Clock* c, double dt) {
    if (threadIdx.x == 0 && blockIdx.x == 0) c->dt = dt;
}

__global__ __launch_bounds__(kDtSlots) void k_set_limits(Clock* c, unsigned long long* slots,
                                                         double max_dt, double limit,
                                                         int reset_scan) {
    if (threadIdx.x == 0) {
        c->max_dt = max_dt;
        c->limit = limit;
    }
    if (reset_scan) slots[threadIdx.x * kDtStride] = 0x7FF0000000000000ull;
}

// ---------------------------------------------------------------------------
// Stores the boundary nodes and ghost layers of q: a thread per (side, layer,
// point) of every axis with a zeroGradient or periodic end, each taking the
// advanced node that stands for its own, so no thread reads what another
// writes.  Layer 0 is the boundary node.  Along x the layers of a row are
// the adjacent doubles, so they are the fastest index there; on the other
// axes x is.
// ---------------------------------------------------------------------------
struct FillCount {
    long long end[3];   // threads of axes 0 .. a
};

__global__ __launch_bounds__(256) void k_fill(GridDev G, double* __restrict__ q, FillCount F,
                                              Fault* fault, long long tag) {
    if (fault->flags) return;
    long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (t >= F.end[2]) return;
    const int axis = t < F.end[0] ? 0 : t < F.end[1] ? 1 : 2;
    if (axis > 0) t -= F.end[axis - 1];
    const int layers = G.g[axis] + 1;
    int p[3], side, l;
    if (axis == 0) {
        l = (int)(t % layers);
        t /= layers;
        side = (int)(t & 1);
        t >>= 1;
        p[1] = (int)(t % G.n[1]);
        p[2] = (int)(t / G.n[1]);
    } else {
        const int o = 3 - axis;
        p[0] = (int)(t % G.n[0]);
        t /= G.n[0];
        p[o] = (int)(t % G.n[o]);
        t /= G.n[o];
        side = (int)(t & 1);
        l = (int)(t >> 1);
    }
    const bool zg = zg_end(G, axis, side);
    if (!zg && (G.wrap[axis] == 0 || l == 0)) return;
    p[axis] = side ? G.n[axis] - 1 + l : -l;
    const long long dst = node_index(G, p[0], p[1], p[2]);
#pragma unroll
    for (int a = 0; a < 3; ++a) {   // the advanced node
        p[a] = map_node(G, a, p[a]);
        if (G.zg_lo[a]) p[a] = max(p[a], G.solved_lo[a]);
        if (G.zg_hi[a]) p[a] = min(p[a], G.solved_hi[a]);
    }
    const long long src = node_index(G, p[0], p[1], p[2]);
    double v5[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) v5[v] = q[v * G.P + src];
    if (zg) {
        const EndEnergy e = end_energy(v5, G.gamma);
        if (l == 0 && !e.ok) raise_fault(kFlagState, &fault->flags, &fault->tag, tag);
        v5[4] = l == 0 ? e.node : e.ghost;
    }
#pragma unroll
    for (int v = 0; v < 5; ++v) q[v * G.P + dst] = v5[v];
}

// Thread per boundary-plane point (2 sides x plane).
template <int AXIS>
__device__ __forceinline__ bool plane_point(const GridDev& G, long long t, int p[3], int& side) {
    constexpr int e1 = (AXIS + 1) % 3, e2 = (AXIS + 2) % 3;
    const long long plane = (long long)G.n[e1] * G.n[e2];
    if (t >= 2 * plane) return false;
    side = (int)(t / plane);
    const long long r = t % plane;
    p[e1] = (int)(r % G.n[e1]);
    p[e2] = (int)(r / G.n[e1]);
    p[AXIS] = side ? G.n[AXIS] - 1 : 0;
    return true;
}

// An end without a condition: its ghost layers take the end node's state
// of src (the state just uploaded) in dst, once; nothing refills them.
template <int AXIS>
__global__ __launch_bounds__(256) void k_bc_hold(GridDev G, const double* __restrict__ src,
                                                 double* __restrict__ dst) {
    int p[3], side;
    const long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (!plane_point<AXIS>(G, t, p, side)) return;
    if (!G.active[AXIS] || G.bc[AXIS] < 2 || zg_end(G, AXIS, side)) return;
    const long long step = G.stride[AXIS];
    const long long b = node_index(G, p[0], p[1], p[2]);
    const long long dir = side ? step : -step;
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        const double val = src[v * G.P + b];
        for (int l = 1; l <= G.g[AXIS]; ++l) dst[v * G.P + b + l * dir] = val;
    }
}

// Clear a fault record (a kernel rather than a memset, so that the clear
// can also be captured in a graph).
__global__ void k_clear_fault(Fault* fault) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        fault->flags = 0u;
        fault->stages = 0u;
        fault->before = 0u;
        fault->tag = -1;
    }
}

// Copy between the caller's unique-node SoA and the padded layout.  A stage
// writes the boundary nodes next to advanced ones only: with `ends` set, a
// node on two or three zeroGradient ends takes the value of the one on the
// first of them.
__global__ __launch_bounds__(256) void k_pack(GridDev G, const double* __restrict__ src,
                                              double* __restrict__ dst, int to_padded,
                                              int ends) {
    const long long N = (long long)G.n[0] * G.n[1] * G.n[2];
    for (long long u = blockIdx.x * (long long)blockDim.x + threadIdx.x; u < N;
         u += (long long)gridDim.x * blockDim.x) {
        const int i = (int)(u % G.n[0]);
        const int j = (int)((u / G.n[0]) % G.n[1]);
        const int k = (int)(u / ((long long)G.n[0] * G.n[1]));
        int p[3] = {i, j, k};
        if (ends) {
            bool on = false;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const int c = min(max(p[a], G.solved_lo[a]), G.solved_hi[a]);
                if (on) p[a] = c;
                on |= p[a] != c;
            }
        }
        const long long id = node_index(G, p[0], p[1], p[2]);
#pragma unroll
        for (int v = 0; v < 5; ++v) {
            if (to_padded) dst[v * G.P + id] = src[v * N + u];
            else dst[v * N + u] = src[v * G.P + id];
        }
    }
}

}  // namespace sfamd
