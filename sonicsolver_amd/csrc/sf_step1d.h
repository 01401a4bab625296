// sf_step1d.h -- a whole physical step of a 1D grid in one launch.
#pragma once

#include "sf_sweep_kernels.h"

namespace sfamd {

// A 1D grid of a few thousand nodes is all latency: a step took a ghost fill
// and an x sweep per stage and a clock launch, 28 us for the 1001 nodes whose
// faces one wave evaluates in 2 us.  Here a block (one wave, one node per
// lane) loads its nodes with a halo of H nodes per stage and side, keeps the
// state in LDS and takes all stages by itself, its valid range shrinking by H
// on each side per stage; it writes the 64 - 2 H stages nodes in the middle.
// The halo is recomputed by the neighbouring blocks (28% of the lanes with
// WENO5 and SSPRK3), which costs nothing while the device has idle SIMDs:
// 200 steps of 1001 nodes take 1.66 ms against 5.57.
//
// Ends: zeroGradient boundary nodes and ghosts are rebuilt in LDS from the
// inner neighbour before every stage, periodic ghosts are nodes like any
// other (loaded a period away), ghosts of an end without a condition keep
// their stored values.  Where the tile holds an end's ghosts, the valid range
// does not shrink on that side.
//
// The clock is kept by the launch, too: dt is the minimum of the CFL
// accumulator that the step before folded into (each block forms it itself),
// block 0 commits the step before and stores dt, and the accumulator of the
// step after is cleared (three are used in turn, so none is cleared or folded
// into while it is read).
constexpr int kStepSets = 3;

struct Step1dArgs {
    GridDev G;
    const double* q;        // step-start state
    double* qout;           // state after the step
    Control* ctl;
    const unsigned long long* scan;   // accumulator holding this step's dt (null: clock.dt)
    unsigned long long* fold;         // ... the next step's CFL scan goes to
    unsigned long long* clear;        // ... to clear
    double* dt_hist;        // may be null
    int slot;
    double cfl;
    long long tag;          // step sequence * 8
};

template <int TIME>
constexpr int step_stages = TIME == 0 ? 1 : TIME == 1 ? 3 : 4;

// Nodes a block of k_step_1d advances.
template <int SCHEME, int TIME>
constexpr int step_nodes = 64 - 2 * (Stencil<SCHEME>::ns / 2) * step_stages<TIME>;

template <int SCHEME, int FLUX, int TIME>
__global__ __launch_bounds__(64) void k_step_1d(Step1dArgs W) {
    constexpr int NS = Stencil<SCHEME>::ns;
    constexpr int H = NS / 2;
    constexpr int ST = step_stages<TIME>;
    constexpr int U = step_nodes<SCHEME, TIME>;
    __shared__ double cur[5][64];
    fetch_args<sizeof(Step1dArgs)>();
    const GridDev& G = W.G;
    Control* const ctl = W.ctl;
    const int t = threadIdx.x;
    const int n = G.n[0];
    const int lo = G.solved_lo[0], hi = G.solved_hi[0];
    const bool periodic = G.wrap[0] != 0;
    const int base = (int)blockIdx.x * U - ST * H;   // node of lane 0
    const int c = base + t;
    // the stored node this lane starts from
    int src = min(max(c, -H), n - 1 + H);
    if (periodic) {
        src = c % n;
        if (src < 0) src += n;
    } else {
        if (G.zg_lo[0]) src = max(src, lo);
        if (G.zg_hi[0]) src = min(src, hi);
    }
    // Everything the step starts from is requested before any of it is waited
    // for: the nodes, the accumulator holding dt, the clock, the fault record.
    // One after the other, three round trips of a microsecond, they were a
    // third of the launch.
    double q[5], q0[5];
    const long long start = node_index(G, src, 0, 0);
#pragma unroll
    for (int v = 0; v < 5; ++v) q0[v] = W.q[v * G.P + start];
    unsigned long long scan = 0;
    if (W.scan) scan = W.scan[t * kDtStride];
    const unsigned fault_flags = ctl->fault.flags;
    const double clock_dt = ctl->clock.dt, max_dt = ctl->clock.max_dt, limit = ctl->clock.limit;
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        q[v] = q0[v];
        cur[v][t] = q[v];
    }
    // A fault of an earlier step, or one that the clock launch before the run
    // found (the CFL scan's and the ghost fill's carry the first step's
    // number): keep the step-start state.  A fault that another block raises
    // in this step does not stop this one, so that the record holds the
    // earliest stage's; which step's it is is read after its flags, as they
    // are published after the tag.
    if (__builtin_expect(fault_flags != 0, 0)) {
        const Fault& f = ctl->fault;
        (void)__hip_atomic_load(&f.flags, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
        const long long tag = __hip_atomic_load(&f.tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (f.before || (tag >> 3) < (W.tag >> 3)) return;
    }
    double dt = clock_dt;
    if (W.scan) {
        dt = __longlong_as_double((long long)wave_min_bits(scan));
        dt = fmin(dt, max_dt);
        dt = fmin(dt, limit);
        if (blockIdx.x == 0 && t == 0) {
            ctl->clock.time += clock_dt;
            ctl->clock.steps += 1;
            ctl->clock.dt = dt;
            if (W.dt_hist) W.dt_hist[W.slot] = dt;
        }
    }
    if (blockIdx.x == 0) W.clear[t * kDtStride] = 0x7FF0000000000000ull;
    const double lw = (FLUX == 5) ? dt / G.d[0] : 0.0;   // Lax-Wendroff dt / spacing
    wave_lds_order();
    // zeroGradient ends held by this tile: lanes outside the advanced range
    // take the last advanced node's state with its rebuilt energy
    const bool from_lo = G.zg_lo[0] && c < lo, from_hi = G.zg_hi[0] && c > hi;
    const int inner = from_lo ? lo - base : from_hi ? hi - base : t;
    unsigned end_flags = 0;
    const auto close_ends = [&] {
        if (from_lo || from_hi) {
            double qi[5];
#pragma unroll
            for (int v = 0; v < 5; ++v) qi[v] = cur[v][inner];
            const EndEnergy e = end_energy(qi, G.gamma);
            end_flags = e.ok ? 0u : kFlagState;
            qi[4] = c == lo - 1 || c == hi + 1 ? e.node : e.ghost;
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                q[v] = qi[v];
                cur[v][t] = qi[v];
            }
        }
        wave_lds_order();
    };
    close_ends();
    // (of the upper zeroGradient ghosts, all equal, the outermost may lie
    // beyond lane 63, which then stands for it)
    const bool fixed_lo = !periodic && base <= -H;
    const bool fixed_hi = !periodic && base + 63 >= n - 1 + H - G.zg_hi[0];
    const bool inside = periodic || (c >= lo && c <= hi);   // a node the steps advance
    // the tile that owns the last advanced node owns the boundary node, too
    const int to = from_hi ? inner : t;
    const bool own = to >= ST * H && to < ST * H + U && c < n;
    // The stages in which this lane's result counts: those that leave its
    // node's stencil whole.  None beyond an end's outer face: lane t's face
    // lies between nodes c and c + 1, those further out are no faces of the
    // grid, and what they raise is nobody's.
    const int whole = min(fixed_lo ? ST : t / H, fixed_hi ? ST : (63 - t) / H);
    const int counted = periodic || (c >= -1 && c < n) ? whole : 0;
    const bool recorded = own || t == ST * H - 1;
    double dt_next = INFINITY;
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};   // RK4: k1 + 2 k2 + 2 k3
#pragma clang loop unroll(disable)
    for (int s = 0; s < ST; ++s) {
        double st[NS][5];
#pragma unroll
        for (int x = 0; x < NS; ++x) {
            const int at = min(max(t + x + 1 - H, 0), 63);
#pragma unroll
            for (int v = 0; v < 5; ++v) st[x][v] = cur[v][at];
        }
        unsigned flags = end_flags;   // of the end closed before this stage
        double f5[5];
        face_flux<0, SCHEME, FLUX>(st, G.gamma, G.area[0], f5, flags, lw);
        if (!finite_sum5(f5)) flags |= kFlagFlux;
        double d5[5];
#pragma unroll
        for (int v = 0; v < 5; ++v) d5[v] = f5[v] - lane_shift_up1(f5[v]);
        if (inside) {
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                const double R = G.jac * d5[v];
                if (TIME == 0) {
                    q[v] = fma(-dt, R, q[v]);
                } else if (TIME == 1) {
                    const double base_w = s == 0 ? 0.0 : s == 1 ? 0.75 : 1.0 / 3.0;
                    const double incr = s == 0 ? 1.0 : s == 1 ? 0.25 : 2.0 / 3.0;
                    q[v] = fma(incr, fma(-dt, R, q[v]), base_w * q0[v]);
                } else if (s < 3) {
                    acc[v] = s == 0 ? R : fma(2.0, R, acc[v]);
                    q[v] = fma(-((s == 2 ? 1.0 : 0.5) * dt), R, q0[v]);
                } else {
                    q[v] = fma(-(dt / 6.0), acc[v] + R, q0[v]);
                }
                cur[v][t] = q[v];
            }
            check_state(q, flags);
            if (s == ST - 1) dt_next = local_dt(G, q, W.cfl, flags);
        }
        // faces and nodes outside the tile's own range count in the tile
        // that owns them; the owner of a boundary node owns its outer face
        const bool raised = s < counted && flags != 0;
        if (raised && recorded) {
            atomicMin((unsigned long long*)&ctl->fault.tag, (unsigned long long)(W.tag + s));
            atomicOr(&ctl->fault.stages, flags << (8 * s));
            __threadfence();
            atomicOr(&ctl->fault.flags, flags);
        }
        // a tile that holds a fault, its own or a neighbour's, stops there:
        // the stages after it would run on what the fault left
        if (__any(raised)) return;
        wave_lds_order();
        close_ends();
    }
    if (end_flags && own) {   // of the end closed after the last stage
        atomicMin((unsigned long long*)&ctl->fault.tag, (unsigned long long)(W.tag + kPhaseFill));
        __threadfence();
        atomicOr(&ctl->fault.flags, end_flags);
    }
    if (own) {
        const long long id = node_index(G, c, 0, 0);
#pragma unroll
        for (int v = 0; v < 5; ++v) W.qout[v * G.P + id] = q[v];
    }
    wave_min_atomic(own && inside ? dt_next : INFINITY, W.fold);
}

// Step of scheme SCHEME with face flux `flux` and time recipe `time`; returns
// -1 for a combination that is not compiled.
template <int SCHEME, int FLUX>
int launch_step1d_f(const Step1dArgs& W, int time, hipStream_t stream) {
    const auto blocks = [&](int nodes) { return (unsigned)((W.G.solved_hi[0] + nodes) / nodes); };
    switch (time) {
    case 0: k_step_1d<SCHEME, FLUX, 0><<<blocks(step_nodes<SCHEME, 0>), 64, 0, stream>>>(W); break;
    case 1: k_step_1d<SCHEME, FLUX, 1><<<blocks(step_nodes<SCHEME, 1>), 64, 0, stream>>>(W); break;
    case 2: k_step_1d<SCHEME, FLUX, 2><<<blocks(step_nodes<SCHEME, 2>), 64, 0, stream>>>(W); break;
    default: return -1;
    }
    return 0;
}

template <int SCHEME>
int launch_step1d(const Step1dArgs& W, int flux, int time, hipStream_t stream) {
    switch (flux) {
    case 0: return launch_step1d_f<SCHEME, 0>(W, time, stream);
    case 1: return launch_step1d_f<SCHEME, 1>(W, time, stream);
    case 2: return launch_step1d_f<SCHEME, 2>(W, time, stream);
    case 3: return launch_step1d_f<SCHEME, 3>(W, time, stream);
    case 4: return launch_step1d_f<SCHEME, 4>(W, time, stream);
    default: return launch_step1d_f<SCHEME, 5>(W, time, stream);
    }
}

extern template int launch_step1d<0>(const Step1dArgs&, int, int, hipStream_t);
extern template int launch_step1d<1>(const Step1dArgs&, int, int, hipStream_t);
extern template int launch_step1d<2>(const Step1dArgs&, int, int, hipStream_t);
extern template int launch_step1d<3>(const Step1dArgs&, int, int, hipStream_t);

}  // namespace sfamd
