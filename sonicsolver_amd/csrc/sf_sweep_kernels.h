// sf_sweep_kernels.h -- the sweep kernels of the grid path: the x sweep
// over flattened face tiles and the y / z march.  Templates only, so every
// translation unit that instantiates a scheme can include it.
#pragma once

#include "sf_device.h"

namespace sfamd {

// ---------------------------------------------------------------------------
// x sweep over the faces of all x lines numbered as one sequence: face
// f = line * (n0 + 1) + (a + 1) lies between nodes a and a+1 of its line
// (a = -1 .. n0-1).  A block is one wave; tile T is faces T*63 .. T*63+63:
// lane t evaluates face T*63+t and lanes 1..63 form the difference for the
// node whose upper face is theirs, taking the lower face's flux from lane
// t-1 by a cross-lane shift (no LDS, no barrier).  Tiles overlap by one
// face, so every node is updated by exactly one lane, and no tile is left
// mostly idle at the end of a line.  Blocks loop over tiles (stride
// gridDim.x), so the CFL fold costs one atomic per block.
// ---------------------------------------------------------------------------
constexpr int kXBlock = 64;

// The x sweeps' arguments, and the wave's own view of them in the kernel
// argument segment.  A sweep has about 90 uniform values (variable pointers,
// grid constants, the ranges of its ends); held across the tile loop they
// exceed the scalar registers, and each restored one costs a v_readlane in
// the loop that the FP64 pipe is waiting for (90 of an x line tile's 880
// vector instructions).  sweep_args() hides where its pointer comes from, so
// that what is read through it is loaded where it is used, by scalar loads
// from the constant cache: 880 -> 800 vector instructions per x line tile
// with WENO5/HLLC.  The 256^3 WENO7/Rusanov x sweep took 919 and takes 779
// us; the 512^3 WENO5/HLLC one keeps its 4.77 ms, in which it moves 21.7 GB,
// 95% of the rate of a large copy.
struct SweepArgs {
    GridDev G;
    const double* q;
    const double* S;
    StageArgs A;
};

__device__ __forceinline__ const SweepArgs& sweep_args() {
    auto p = (const __attribute__((address_space(4))) SweepArgs*)
        __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const SweepArgs*)p;
}

// Requests every 64-byte line of a kernel's first BYTES of arguments and waits
// for them once.  Read where they are needed, the arguments of a stage arrive
// in three or four round trips to memory, each for lines that no wave of the
// compute unit has read yet, before the first node is requested.  For kernels
// that are all latency: 200 steps of 1001 nodes 1.69 -> 1.65 ms, 20 of 193 x
// 97 0.563 -> 0.548; k_stage_yx on 853^2 gained nothing (2.831, 2.836).
template <int BYTES>
__device__ __forceinline__ void fetch_args() {
    const auto p = (const __attribute__((address_space(4))) unsigned*)
        __builtin_amdgcn_kernarg_segment_ptr();
    unsigned x = 0;
#pragma unroll
    for (int b = 0; b < BYTES; b += 64) x |= p[b / 4];
    asm volatile("" ::"s"(x));
}

// The value of lane t-1 (lane 0 receives 0): one DPP wave shift per 32-bit
// half, a VALU move with no LDS round trip.
__device__ __forceinline__ double lane_shift_up1(double x) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffll), 0x138, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x138, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// The value of lane 63, as a wave-uniform value.
__device__ __forceinline__ double lane63(double x) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), 63);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// The double `nodes` past base + off bytes: a uniform base, a lane's 32-bit
// byte offset and a constant, which one load instruction takes as they are.
__device__ __forceinline__ double at(const double* base, unsigned off, int nodes = 0) {
    return *(const double*)((const char*)base + off + 8 * nodes);
}

// The final sweep's operands for the node `off` bytes past node id0: its
// current value, the flux difference the y and z sweeps accumulated and its
// step-start value.  All three are loaded for every lane, without a test:
// every lane's node index lies in the padded grid (a lane without a node of
// its own takes the tile's first); on a grid without a y axis no sweep
// writes S, which keeps the zeros it was created with, so its sum is the x
// difference alone; where the recipe does not read q0 (Euler, the first
// SSPRK3 stage) the values go unused, and there q0 is the stage input
// itself, so the loads hit the lines the stencil loads bring in.
__device__ __forceinline__ void stage_operands(long long id0, unsigned off, double (&pq)[5],
                                               double (&ps)[5], double (&pq0)[5]) {
    const SweepArgs& W = sweep_args();
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        pq[v] = at(W.q + v * W.G.P + id0, off);
        ps[v] = at(W.S + v * W.G.P + id0, off);
        pq0[v] = at(W.A.q0 + v * W.G.P + id0, off);
    }
}

// Three waves per SIMD: the registers that hold the final sweep's stage
// operands through the face arithmetic pay more than a fourth wave would
// (and four would spill).
// The x sweep is always a stage's last sweep (x is always active and the
// sweeps run z, y, x), so it always applies the stage update.  TIME: the
// time recipe (A.time, fixed at compile time so that the update carries no
// code for the other recipes).
template <int SCHEME, int FLUX, int TIME>
__global__ __launch_bounds__(kXBlock)
__attribute__((amdgpu_waves_per_eu(3, 8))) void k_sweep_x(SweepArgs W) {
    if (*W.A.flags) return;   // a fault was raised: keep the step-start state
    // face numbers fit 32 bits: the host rejects grids with 2^32 - 2^8
    // faces or more along x
    const int t = threadIdx.x;
    const unsigned per_line = W.G.n[0] + 1;
    const unsigned faces = per_line * W.G.n[1] * W.G.n[2];
    const unsigned tiles = (faces - 1 + kXBlock - 2) / (kXBlock - 1);
    unsigned flags = 0;
    double dt_local = INFINITY;
    const double dt_step = TIME == 3 ? 0.0 : *W.A.dt;   // the step's dt, read once
    const double lw = (FLUX == 5) ? *W.A.dt / W.G.d[0] : 0.0;   // Lax-Wendroff dt / spacing
    // Blocks are dealt to the 8 XCDs round-robin (block b runs on XCD b % 8),
    // each with its own L2; tiles are numbered so that the blocks of one XCD
    // take consecutive tiles and share the stencil halo between them in that
    // L2.  The grid size is a multiple of 8.
    const unsigned per_xcd = gridDim.x >> 3;
    const unsigned first = (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3);
    for (unsigned T = first; T < tiles; T += gridDim.x) {
        const SweepArgs& F = sweep_args();
        const GridDev& G = F.G;
        const unsigned f = T * (kXBlock - 1) + t;
        const bool face = f < faces;
        const unsigned line = face ? fast_div(f, G.div_line) : 0;
        const int a = face ? (int)(f - line * per_line) - 1 : 0;  // lower node of the face
        const unsigned kz = fast_div(line, G.div_n1);
        const int j = (int)(line - kz * (unsigned)G.n[1]), k = (int)kz;
        double f5[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        // A tile's nodes lie within a few lines, in ascending order, so a
        // lane addresses its node by a 32-bit offset from the first lane's.
        // The final sweep's stage operands for the node this lane updates
        // (the lower node of its face) are loaded before the face
        // arithmetic, so that their latency hides behind it -- except for
        // WENO7, whose eight-node stencil leaves no registers to hold them at
        // three waves per SIMD; it loads them after the face.
        const bool upd = t >= 1 && face && a >= 0;
        const unsigned uid = (unsigned)node_index(G, a, j, k);
        const unsigned id0 = __builtin_amdgcn_readfirstlane(uid);
        const unsigned off = face ? (uid - id0) * 8u : 0u;
        double pq[5], ps[5], pq0[5];
        constexpr bool kEarly = SCHEME != 3;
        if (kEarly) stage_operands(id0, off, pq, ps, pq0);
        if (face) {
            constexpr int NS = Stencil<SCHEME>::ns;
            double st[NS][5];
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                const double* row = F.q + v * G.P + id0;
#pragma unroll
                for (int s = 0; s < NS; ++s) st[s][v] = at(row, off, s + 1 - NS / 2);
            }
            face_flux<0, SCHEME, FLUX>(st, G.gamma, G.area[0], f5, flags, lw);
            if (!finite_sum5(f5)) flags |= kFlagFlux;
        }
        double lower[5];
#pragma unroll
        for (int v = 0; v < 5; ++v) lower[v] = lane_shift_up1(f5[v]);
        if (upd) {
            const SweepArgs& U = F;
            if (!kEarly) stage_operands(id0, off, pq, ps, pq0);
            const long long id = uid;
            double s5[5];
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                const double d = f5[v] - lower[v];
                s5[v] = ps[v] + d;
            }
            double dl = INFINITY;
            double qn[5];
            if (solved_node(U.G, a, j, k)) {
                stage_update_dt<TIME>(U.G, U.A, id, pq, pq0, s5, dt_step, flags, dl, qn);
            } else if (TIME != 3) {
#pragma unroll
                for (int v = 0; v < 5; ++v) {
                    qn[v] = pq[v];   // not advanced: carried over
                    U.A.qout[v * U.G.P + id] = qn[v];
                }
            }
            dt_local = fmin(dt_local, dl);
        }
    }
    raise_fault(flags, W.A.flags, W.A.fault_tag, W.A.tag);
    if (W.A.reduce_dt) wave_min_atomic(dt_local, W.A.dtmin);
}

// ---------------------------------------------------------------------------
// x sweep by whole lines, for grids with many x lines: a block (one wave)
// takes groups of kLineGroup lines and walks each line in tiles of 64
// nodes, lane t evaluating the upper face of node 64m + t; node 64m + t
// takes its lower face from lane t-1 by the cross-lane shift, lane 0 from
// the previous tile's lane 63 (kept in scalar registers), and the first
// tile of a line from the line's first face, which the group evaluates for
// its lines at once before walking them.  Rows start on 128-byte lines, so
// a tile's loads and stores are whole lines.  Every node takes the same
// faces and the same arithmetic as in k_sweep_x, so the two give identical
// results.
//
// All loads go through LDS by 16-byte global-to-LDS copies, which the
// memory pipe completes while the wave computes: the conserved variables
// of the next tile with a halo of four nodes on each side (72 per
// variable, two buffers used in turn) are requested before the current
// tile's faces, and the current tile's S and q0 (one 64-node row each,
// lanes 0-31 one variable and 32-63 the next, two nodes per lane) before
// its update.  The stencils are read from LDS, so the face arithmetic
// never waits for memory and no register holds an operand across it.  The
// copies are not counted by the compiler for LDS reads: one explicit wait
// for the vector memory count to reach zero, after the faces, covers both
// the tile's S, q0 and the next tile's variables (all requested before it).
// ---------------------------------------------------------------------------
constexpr int kLineGroup = 8;   // 16 ran 1-2.5% slower on 256^3, the same on 512^3
constexpr int kHalo = 4;                      // nodes each side of a tile
constexpr int kRow = kXBlock + 2 * kHalo;     // 72 doubles per variable
constexpr int kRowLanes = kRow / 2;           // lanes of 16 bytes per row

template <int SCHEME, int FLUX, int TIME>
__global__ __launch_bounds__(kXBlock)
__attribute__((amdgpu_waves_per_eu(3, 8))) void k_sweep_xl(SweepArgs W) {
    if (*W.A.flags) return;   // a fault was raised: keep the step-start state
    constexpr int NS = Stencil<SCHEME>::ns;
    static_assert(NS / 2 <= kHalo, "the halo covers the stencil");
    __shared__ double first[5][kLineGroup];   // each line's face -1/2
    __shared__ __attribute__((aligned(16))) double qb[2][5][kRow];
    __shared__ __attribute__((aligned(16))) double pk[10][kXBlock];   // S 0-4, q0 5-9
    const int t = threadIdx.x;
    const int n0 = W.G.n[0];
    const unsigned lines = (unsigned)W.G.n[1] * (unsigned)W.G.n[2];
    const unsigned groups = (lines + kLineGroup - 1) / kLineGroup;
    const int tiles = (n0 + kXBlock - 1) / kXBlock;
    const int last_needed = n0 - 1 + NS / 2;   // the highest node a stencil reads
    // S / q0 copies: byte offset of this lane's two nodes in the lower
    // variable of a copy, and of the upper variable (P doubles further;
    // the host keeps 8 P + 1024 below 2^32)
    const int pair = t & 31;
    const unsigned up = (t >> 5) ? (unsigned)W.G.P * 8u : 0u;
    unsigned flags = 0;
    double dt_local = INFINITY;
    const double dt_step = TIME == 3 ? 0.0 : *W.A.dt;   // the step's dt, read once
    const double lw = (FLUX == 5) ? *W.A.dt / W.G.d[0] : 0.0;   // Lax-Wendroff dt / spacing

    // the 72 nodes 64m-4 .. 64m+67 of line (j, k), all five variables, into
    // buffer b; lanes 0-35 take two nodes each, a lane whose first node no
    // stencil reads copies the row's first two again (the second node of a
    // pair is at most one past the last ghost, which every row holds)
    auto fetch_q = [&](int b, int m, int j, int k) {
        if (t < kRowLanes) {
            const SweepArgs& T = sweep_args();
            const int node0 = m * kXBlock - kHalo;
            const long long id = node_index(T.G, node0, j, k);
            const unsigned off = (node0 + 2 * t <= last_needed ? (unsigned)t : 0u) * 16u;
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                const char* base = (const char*)(T.q + v * T.G.P + id);
                __builtin_amdgcn_global_load_lds(
                    (__attribute__((address_space(1))) void*)(base + off),
                    (__attribute__((address_space(3))) void*)&qb[b][v][0], 16, 0, 0);
            }
        }
    };
    auto wait_copies = [] {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
        __builtin_amdgcn_sched_barrier(0);
    };

    for (unsigned grp = blockIdx.x; grp < groups; grp += gridDim.x) {
        const unsigned line0 = grp * kLineGroup;
        const unsigned nl = min((unsigned)kLineGroup, lines - line0);
        const SweepArgs& W1 = sweep_args();
        const GridDev& G = W1.G;
        const int n1 = G.n[1];
        int j, k;
        {
            const unsigned kz = fast_div(line0, G.div_n1);
            j = (int)(line0 - kz * (unsigned)G.n[1]);
            k = (int)kz;
        }
        fetch_q(0, 0, j, k);   // the group's first tile
        // the first face (-1/2) of the group's lines, lane l for line0 + l
        {
            const unsigned line = line0 + (unsigned)t;
            if (t < kLineGroup && line < lines) {
                const unsigned kz = fast_div(line, G.div_n1);
                const int jl = (int)(line - kz * (unsigned)G.n[1]), kl = (int)kz;
                const long long id = node_index(G, -1, jl, kl);
                double st[NS][5];
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int v = 0; v < 5; ++v) st[s][v] = W1.q[v * G.P + id + (s + 1 - NS / 2)];
                double f5[5];
                face_flux<0, SCHEME, FLUX>(st, G.gamma, G.area[0], f5, flags, lw);
                if (!finite_sum5(f5)) flags |= kFlagFlux;
#pragma unroll
                for (int v = 0; v < 5; ++v) first[v][t] = f5[v];
            }
        }
        wait_copies();
        __syncthreads();
        int b = 0;   // the buffer holding the current tile's variables
        for (unsigned l = 0; l < nl; ++l) {
            double carry[5];
#pragma unroll
            for (int v = 0; v < 5; ++v) carry[v] = first[v][l];
            for (int m = 0; m < tiles; ++m) {
                const int a = m * kXBlock + t;   // this lane's node
                const int rem = n0 - m * kXBlock;
                const bool node = t < rem;
                const SweepArgs& T = sweep_args();
                const long long id0 = node_index(T.G, m * kXBlock, j, k);
                // the next tile's variables (next line's first tile at the
                // end of a line, none after the group's last)
                {
                    int jn = j, kn = k, mn = m + 1;
                    bool more = true;
                    if (mn == tiles) {
                        mn = 0;
                        more = l + 1 < nl;
                        if (++jn == n1) { jn = 0; ++kn; }
                    }
                    if (more) fetch_q(b ^ 1, mn, jn, kn);
                }
                // this tile's S and q0; a lane whose nodes lie past the
                // line's end copies the tile's first two again
                {
                    const unsigned lo = (unsigned)(2 * pair < rem ? pair : 0) * 16u;
                    const double* const src[2] = {T.S, T.A.q0};
#pragma unroll
                    for (int c = 0; c < 6; ++c) {
                        const int arr = c / 3, v = 2 * (c % 3);
                        if (v < 4 || t < 32) {
                            const char* base = (const char*)(src[arr] + v * T.G.P + id0);
                            const unsigned off = lo + (v < 4 ? up : 0u);
                            __builtin_amdgcn_global_load_lds(
                                (__attribute__((address_space(1))) void*)(base + off),
                                (__attribute__((address_space(3))) void*)&pk[5 * arr + v][0], 16, 0,
                                0);
                        }
                    }
                }
                // the stencil from LDS (lanes past the line's end take the
                // last node's)
                const int ti = node ? t : rem - 1;
                double st[NS][5];
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int v = 0; v < 5; ++v) st[s][v] = qb[b][v][ti + kHalo + s + 1 - NS / 2];
                double f5[5];
                face_flux<0, SCHEME, FLUX>(st, T.G.gamma, T.G.area[0], f5, flags, lw);
                if (!finite_sum5(f5)) flags |= kFlagFlux;
                double lower[5];
#pragma unroll
                for (int v = 0; v < 5; ++v) {
                    const double sh = lane_shift_up1(f5[v]);
                    lower[v] = t == 0 ? carry[v] : sh;
                    carry[v] = lane63(f5[v]);   // the next tile's first lower face
                }
                wait_copies();
                if (node) {
                    const SweepArgs& U = sweep_args();
                    const long long id = id0 + t;
                    double pq[5], ps[5], pq0[5];
#pragma unroll
                    for (int v = 0; v < 5; ++v) {
                        pq[v] = qb[b][v][t + kHalo];
                        ps[v] = pk[v][t];
                        pq0[v] = pk[5 + v][t];
                    }
                    double s5[5];
#pragma unroll
                    for (int v = 0; v < 5; ++v) {
                        const double d = f5[v] - lower[v];
                        s5[v] = ps[v] + d;
                    }
                    double dl = INFINITY;
                    double qn[5];
                    if (solved_node(U.G, a, j, k)) {
                        stage_update_dt<TIME>(U.G, U.A, id, pq, pq0, s5, dt_step, flags, dl, qn);
                    } else if (TIME != 3) {
#pragma unroll
                        for (int v = 0; v < 5; ++v) {
                            qn[v] = pq[v];   // not advanced: carried over
                            U.A.qout[v * U.G.P + id] = qn[v];
                        }
                    }
                    dt_local = fmin(dt_local, dl);
                }
                b ^= 1;
            }
            if (++j == n1) { j = 0; ++k; }
        }
        __syncthreads();
    }
    raise_fault(flags, W.A.flags, W.A.fault_tag, W.A.tag);
    if (W.A.reduce_dt) wave_min_atomic(dt_local, W.A.dtmin);
}

// ---------------------------------------------------------------------------
// y / z sweep over the advanced nodes: lane = x index, blockIdx.y = the
// remaining transverse index, blockIdx.z = segment of SEG nodes along the
// sweep axis.  Each lane marches
// along its column; the NS-node stencil window lives in LDS (one private
// slot set per lane, a ring indexed by `head`), so between faces only the
// previous face flux stays in registers.  Lanes never read each other's
// slots, so no barrier is needed.
// ---------------------------------------------------------------------------
constexpr int kMarchBlock = 64;

// The WENO5 ring (10 KB per wave) leaves room for four waves per SIMD; the
// register count decides how many run: the WENO5, TENO5 and WENO3 marches
// with the Rusanov or HLLC flux fit 128 registers and run four, the other
// fluxes' need a few more and run three (holding them to 128 spills).
// Bound by FP64 issue.  On 512^3 with WENO5/HLLC the z / y march took 4.03 /
// 4.33 ms; 3.51 / 3.90 with the shorter face arithmetic and the face's two
// nodes read from the ring again after the reconstruction (120 registers;
// held across it they cost the fourth wave); 3.41 / 3.71 with the y march's
// sums requested before the Riemann solver and without the wait for the
// previous node's stores at the head of the loop.
template <int AXIS, int SCHEME, int FLUX, int MODE>
__global__ __launch_bounds__(kMarchBlock)
void k_sweep_march(GridDev G,
                                                             const double* __restrict__ q,
                                                             double* __restrict__ S, StageArgs A,
                                                             int seg) {
    constexpr int NS = Stencil<SCHEME>::ns;
    constexpr int H = NS / 2;    // face a+1/2 reads nodes a+1-H .. a+H
    constexpr int W = NS - 2;    // LDS ring slots: nodes a+1-H .. a+H-2
    __shared__ double win[W][5][kMarchBlock];
    const int lane = threadIdx.x;
    // Only advanced nodes need a sum, so the march covers their ranges; along
    // x a boundary node takes the sum of the node next to it, because S has
    // to be written without holes: with node 0 of every row left out, the
    // 201 x 87 x 45 z march took 80 us instead of 38.  Blocks start on
    // 128-byte lines.
    const int i = blockIdx.x * kMarchBlock + lane;
    const int ic = min(max(i, G.solved_lo[0]), G.solved_hi[0]);
    const int o = G.solved_lo[3 - AXIS] + blockIdx.y;
    const int a0 = G.solved_lo[AXIS] + blockIdx.z * seg;
    const int a1 = min(a0 + seg, G.solved_hi[AXIS] + 1);
    static_assert(MODE == kCopyS || MODE == kAccumS, "a march writes or accumulates S; the x sweep applies the update");
    const unsigned raised = *A.flags;   // tested once the window is on its way
    unsigned flags = 0;
    const double lw = (FLUX == 5) ? StepClock(A).get(A) / G.d[AXIS] : 0.0;   // dt / spacing
    if (i < G.n[0]) {
        const long long step = G.stride[AXIS];
        // The face a+1/2 reads its NS nodes as W from the lane's LDS ring
        // (nodes a+1-H .. a+H-2), node a+H-1 carried in registers from the
        // previous face and node a+H loaded for this face.  The march starts
        // one node early (a = a0-1) so that face a0-1/2 is evaluated by the
        // same instructions as every other face: a face's rounding then does
        // not depend on where a segment starts.
        const long long col = node_index(G, ic, AXIS == 1 ? 0 : o, AXIS == 2 ? 0 : o);
        const auto node = [&](int a) { return col + map_node(G, AXIS, a) * step; };
        long long id = col + (i - ic) + (a0 - 1) * step;   // node a
        for (int s = 0; s < W; ++s)
#pragma unroll
            for (int v = 0; v < 5; ++v) win[s][v][lane] = q[v * G.P + node(a0 - H + s)];
        double carried[5];
#pragma unroll
        for (int v = 0; v < 5; ++v) carried[v] = q[v * G.P + node(a0 + H - 2)];
        int head = 0;          // slot of the oldest node
        double fprev[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        // Pinned, so that the wait for the carried node stands here and not at
        // the head of the loop, where it would also wait for the stores of
        // the previous node.
#pragma unroll
        for (int v = 0; v < 5; ++v) asm volatile("" : "+v"(carried[v]));
        if (raised) return;   // a fault was raised: keep the step-start state
#pragma clang loop unroll(disable)
        for (int a = a0 - 1; a < a1; ++a, id += step) {
            double st[NS][5];
#pragma unroll
            for (int v = 0; v < 5; ++v) st[NS - 1][v] = q[v * G.P + node(a + H)];
#pragma unroll
            for (int s = 0; s < W; ++s) {
                const int slot = (head + s >= W) ? head + s - W : head + s;
#pragma unroll
                for (int v = 0; v < 5; ++v) st[s][v] = win[slot][v][lane];
            }
            // the oldest node leaves the ring, the carried one enters it
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                st[NS - 2][v] = carried[v];
                win[head][v][lane] = carried[v];
                carried[v] = st[NS - 1][v];
            }
            head = (head == W - 1) ? 0 : head + 1;
            // the face's two nodes a and a+1: ring slots H-1 and H of the
            // window as it was (slots H-2 and H-1 from the new head); for
            // WENO3, whose ring holds two nodes, the right one is the node
            // that just entered.  The sum this face's difference is added to
            // is requested here too, so that the Riemann solver hides its
            // latency (the node a0 - 1, whose sum goes unused, lies in the
            // padded grid).
            double sold[5];
            const auto base = [&](int side, double (&b)[5]) {
                if (MODE == kAccumS && side == 0) {
#pragma unroll
                    for (int v = 0; v < 5; ++v) sold[v] = S[v * G.P + id];
                }
                const int s = H - 2 + side;
                const int slot = (head + s >= W) ? head + s - W : head + s;
#pragma unroll
                for (int v = 0; v < 5; ++v) b[v] = win[slot][v][lane];
            };
            double f[5];
            face_flux_from<AXIS, SCHEME, FLUX>(st, base, G.gamma, G.area[AXIS], f, flags, lw);
            double s5[5];
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                if (!isfinite(f[v])) flags |= kFlagFlux;
                s5[v] = f[v] - fprev[v];
                fprev[v] = f[v];
            }
            if (MODE == kAccumS) {
                // pinned, so that the loads of sold stay where they are
#pragma unroll
                for (int v = 0; v < 5; ++v) {
                    s5[v] = sold[v] + s5[v];
                    asm volatile("" : "+v"(s5[v]));
                }
            }
            if (a < a0) continue;
#pragma unroll
            for (int v = 0; v < 5; ++v) S[v * G.P + id] = s5[v];
        }
    }
    raise_fault(flags, A.flags, A.fault_tag, A.tag);
}

// ---------------------------------------------------------------------------
// y and x faces and the stage update of the advanced nodes in one march along
// y: a wave takes 64 columns of one z plane and up to kYxRows rows, and a
// block one wave or kYxWaves of them, one above the other.  Ghosts are read through map_node (a lane's column and a row's
// number are mapped once each), and next to a zeroGradient end the launch
// writes the boundary node and first ghost of what it advances, so no ghost
// fill is needed between stages.  At row a
// every lane evaluates its upper y face from its own column, as
// k_sweep_march does, and its upper x face from the same row of the LDS
// ring, whose rows carry the NS - 1 halo columns the x stencils reach; the
// lower x face comes from lane t-1 by the cross-lane shift.  Lane 0 takes it
// from the block's first faces, which the lanes evaluate beforehand, one row
// each (cols = 64), or is itself only there to evaluate it (cols = 63, the
// blocks overlapping by a column).  Faces, sums and updates are formed by
// the same functions in the same order as by the separate sweeps, so the
// results are theirs bit for bit.
//
// Against the y march and the x sweep it neither writes nor reads back the
// y differences and reads the state once: on 512^3 27.3 GB per launch instead
// of 16.6 + 21.6 (7.6 ms instead of 3.7 + 4.8).  Bound by FP64 issue (87% of
// the cycles, 86% of it FP64) at three waves per SIMD (two for
// WENO7, whose ring is 17 KB).  yx_shape chooses the rows and columns.
// ---------------------------------------------------------------------------
constexpr int kYxRows = 32;
constexpr int kYxWaves = 4, kYxWaveRows = 8;   // blocks of several waves

// Node (i, j, k) at id was advanced to qn: next to a zeroGradient end, write
// the boundary node and the first ghost layer (which stands for the others,
// map_node).  Raises kFlagState where the end's pressures are not positive,
// which check_state's test of qn decides alike except where the internal
// energy is within some ulps of the kinetic energy.  RUN: only where no check
// is raised already, which stops a grid's run; a batch's problem finishes its
// step.
// Filling the ghosts by launches of their own took four 4-5 us launches per
// stage in 2D and six in 3D, latency alone: a pass of 20 steps on 853^2 takes
// 3.51 ms without them and 4.31 with, on 193 x 97 0.83 and 1.87.
template <bool CORNERS = false, bool RUN = !CORNERS>
__device__ __forceinline__ void write_ends(const GridDev& G, double* __restrict__ out, int i,
                                           int j, int k, long long id, const double qn[5],
                                           unsigned& flags) {
    const int c[3] = {i, j, k};
    bool at_end = false;
#pragma unroll
    for (int a = 0; a < 3; ++a)
        at_end |= (G.zg_lo[a] && c[a] == G.solved_lo[a]) || (G.zg_hi[a] && c[a] == G.solved_hi[a]);
    if (!at_end) return;
    const EndEnergy e = end_energy(qn, G.gamma);
    if (!e.ok && !(RUN && flags)) flags |= kFlagState;
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int side = 0; side < 2; ++side) {
            const bool here = side ? G.zg_hi[a] && c[a] == G.solved_hi[a]
                                   : G.zg_lo[a] && c[a] == G.solved_lo[a];
            if (!here) continue;
            const long long dir = side ? G.stride[a] : -G.stride[a];
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                out[v * G.P + id + dir] = v == 4 ? e.node : qn[v];
                out[v * G.P + id + 2 * dir] = v == 4 ? e.ghost : qn[v];
            }
        }
    if (CORNERS) {   // of a plane whose four ends carry zeroGradient
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int sx = c & 1, sy = c >> 1;
            const bool here = i == (sx ? G.solved_hi[0] : G.solved_lo[0]) &&
                              j == (sy ? G.solved_hi[1] : G.solved_lo[1]) && G.zg_lo[1];
            if (!here) continue;
            const long long at = id + (sx ? 1 : -1) + (sy ? G.stride[1] : -G.stride[1]);
#pragma unroll
            for (int v = 0; v < 5; ++v) out[v * G.P + at] = v == 4 ? e.node : qn[v];
        }
    }
}

// Orders the LDS accesses of a wave's lanes among themselves: the hardware
// performs a wave's LDS operations in order, so only the compiler has to
// keep them so.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct YxShape {
    int cols;      // columns a block advances: 64, or 63 with a helper lane
    int rows;      // rows a wave advances (at most kYxRows), of a block of
    int waves;     // this many waves (1 or kYxWaves)
    int nx, ny;    // blocks along x and along y
    unsigned blocks;
    int block;     // 1: a wave per face (k_block_yx)
};

// LDS of a block that advances a tile of a y / x stage.
template <int SCHEME, int WAVES = 1>
struct YxLds {
    static constexpr int NS = Stencil<SCHEME>::ns;
    static constexpr int rows = WAVES > 1 ? kYxWaveRows : kYxRows;
    double win[WAVES][NS - 2][5][kXBlock + NS];   // ring rows a+1-H .. a+H-2, each
                                                  // H-1 halo columns, 64, H halo, 1 pad
    double first[WAVES][5][rows];
    double edge[WAVES > 1 ? WAVES - 1 : 1][5][WAVES > 1 ? kXBlock : 1];
};

// One wave's tile: rows a0 .. a1-1 of plane k; lane t has column i0 + t.  W
// and args() are the sweep's arguments, args() as sweep_args() reads them.
// CORNERS: write_ends writes the corners, too; SLOTS: partial minima of the
// CFL accumulator.  The waves of a block (WAVES > 1) lie one above the other:
// the last y face of each is the first of the next, which is evaluated there,
// at the start of the march, and passed on in LDS.
template <int SCHEME, int FLUX, int TIME, bool HAS_S, bool CORNERS, int SLOTS, int WAVES, class Args>
__device__ __forceinline__ void stage_yx_tile(const SweepArgs& W, const Args& args,
                                              YxLds<SCHEME, WAVES>& lds, int i0, int helper,
                                              int a0, int a1, int k, bool first_block,
                                              unsigned raised) {
    constexpr int NS = Stencil<SCHEME>::ns;
    constexpr int H = NS / 2;
    constexpr int R = NS - 2;
    constexpr int HC = NS - 1;            // halo columns per row and variable
    static_assert(5 * HC <= kXBlock, "one lane per halo value");
    const int w = WAVES > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / kXBlock) : 0;
    auto& win = lds.win[w];
    auto& first = lds.first[w];
    const int t = WAVES > 1 ? threadIdx.x & (kXBlock - 1) : threadIdx.x;
    const int i = i0 + t;
    const int hi0 = W.G.solved_hi[0];
    if (WAVES > 1 && a0 >= a1) {   // no rows left for this wave
        __syncthreads();
        return;
    }
    const bool edge = WAVES > 1 && w < WAVES - 1 && a1 <= W.G.solved_hi[1];
    // this lane advances node i (none of a block's waves leaves early where
    // a fault was raised, because the others may have read the flags before)
    const bool node = i <= hi0 && t >= helper && !(WAVES > 1 && raised);
    const int last = hi0 + H;                          // the last column a face reads
    unsigned flags = 0;
    double dt_local = INFINITY;
    const StepClock clock(W.A);
    const double dt_lw = (FLUX == 5) ? clock.get(W.A) : 0.0;
    const double lwx = (FLUX == 5) ? dt_lw / W.G.d[0] : 0.0;   // Lax-Wendroff dt / spacing
    const double lwy = (FLUX == 5) ? dt_lw / W.G.d[1] : 0.0;
    // Rows are addressed from their first double (column -xo) by a lane's
    // 32-bit byte offset.
    const int xo = W.G.xo;
    const auto row_of = [&](const GridDev& G, int a) {
        return node_index(G, -xo, map_node(G, 1, a), k);
    };

    // the block's first x faces (lower face of lane 0's node), lane r for
    // row a0 + r
    if (helper == 0 && a0 + t < a1) {
        const long long row = row_of(W.G, a0 + t);
        double st[NS][5];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int c = map_node(W.G, 0, i0 - H + s) + xo;
#pragma unroll
            for (int v = 0; v < 5; ++v) st[s][v] = W.q[v * W.G.P + row + c];
        }
        double f5[5];
        face_flux<0, SCHEME, FLUX>(st, W.G.gamma, W.G.area[0], f5, flags, lwx);
        if (!finite_sum5(f5)) flags |= kFlagFlux;
#pragma unroll
        for (int v = 0; v < 5; ++v) first[v][t] = f5[v];
    }

    // Lanes past the last column load it again and form faces that nothing
    // takes.
    const unsigned off = (unsigned)(map_node(W.G, 0, min(i, last)) + xo) * 8u;
    // halo: lane l < 5 HC loads variable l / HC, halo column l % HC
    const int hv = t / HC, hc = t % HC;
    const bool halo = hv < 5;
    const int hcol = hc < H - 1 ? hc - (H - 1) : kXBlock + hc - (H - 1);   // from i0
    const double* hsrc =
        W.q + (halo ? hv : 0) * W.G.P + (map_node(W.G, 0, min(i0 + hcol, last)) + xo);
    const int hpos = hcol + H - 1;
    const long long step = W.G.stride[1];
    const unsigned own = (unsigned)(i + xo) * 8u;   // the lane's own node, where it has one
    for (int s = 0; s < R; ++s) {
        const long long row = row_of(W.G, a0 - H + s);
#pragma unroll
        for (int v = 0; v < 5; ++v) win[s][v][t + H - 1] = at(W.q + v * W.G.P + row, off);
    }
    double carried[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) carried[v] = at(W.q + v * W.G.P + row_of(W.G, a0 + H - 2), off);
#pragma unroll
    for (int v = 0; v < 5; ++v) asm volatile("" : "+v"(carried[v]));
    double hnext = 0.0;
    int head = 0;
    double fprev[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    long long id = node_index(W.G, -xo, a0 - 1, k);   // row a
    wave_lds_order();
    const double dt_step = clock.get(W.A);
    if (first_block) clock.commit(W.A, dt_step);
    if (WAVES == 1 && raised) return;   // a fault was raised: keep the step-start state
#pragma clang loop unroll(disable)
    for (int a = a0 - 1; a < a1; ++a, id += step) {
        const SweepArgs& T = args();
        // the halo columns of row a join the ring; those of row a + 1 are
        // requested
        const auto slot = [&](int s) { return (head + s >= R) ? head + s - R : head + s; };
        if (halo) {
            win[slot(H - 1)][hv][hpos] = hnext;
            hnext = hsrc[row_of(T.G, a + 1)];
        }
        double st[NS][5];
#pragma unroll
        for (int v = 0; v < 5; ++v) st[NS - 1][v] = at(T.q + v * T.G.P + row_of(T.G, a + H), off);
#pragma unroll
        for (int s = 0; s < R; ++s)
#pragma unroll
            for (int v = 0; v < 5; ++v) st[s][v] = win[slot(s)][v][t + H - 1];
#pragma unroll
        for (int v = 0; v < 5; ++v) {
            st[NS - 2][v] = carried[v];
            win[head][v][t + H - 1] = carried[v];
            carried[v] = st[NS - 1][v];
        }
        head = (head == R - 1) ? 0 : head + 1;
        wave_lds_order();
        // rows a and a + 1 are now at H - 2 and H - 1 from the head
        const int ra = slot(H - 2), rb = slot(H - 1);
        unsigned fy = 0;
        double s5[5];
        {
            double f[5];
            if (edge && a == a1 - 1) {
#pragma unroll
                for (int v = 0; v < 5; ++v) f[v] = lds.edge[WAVES > 1 ? w : 0][v][t];
            } else {
                face_flux_from<1, SCHEME, FLUX>(
                    st,
                    [&](int side, double (&b)[5]) {
#pragma unroll
                        for (int v = 0; v < 5; ++v) b[v] = win[side ? rb : ra][v][t + H - 1];
                    },
                    T.G.gamma, T.G.area[1], f, fy, lwy);
                if (!finite5(f)) fy |= kFlagFlux;
            }
            if (WAVES > 1 && a < a0) {
                if (w > 0) {
#pragma unroll
                    for (int v = 0; v < 5; ++v) lds.edge[w - 1][v][t] = f[v];
                }
                __syncthreads();
            }
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                s5[v] = f[v] - fprev[v];
                fprev[v] = f[v];
            }
        }
        if (node) flags |= fy;
        if (a < a0) continue;
        // the x face; the stage operands are requested before its Riemann
        // solver, which hides their latency
        double sx[NS][5], ps[5], pq0[5], f5[5];
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int v = 0; v < 5; ++v) sx[s][v] = win[ra][v][t + s];
        unsigned fx = 0;
        face_flux_from<0, SCHEME, FLUX>(
            sx,
            [&](int side, double (&b)[5]) {
                if (side == 0) {
                    const SweepArgs& U = args();
#pragma unroll
                    for (int v = 0; v < 5; ++v) {
                        if (HAS_S) ps[v] = at(U.S + v * U.G.P + id, node ? own : off);
                        pq0[v] = at(U.A.q0 + v * U.G.P + id, node ? own : off);
                    }
                }
#pragma unroll
                for (int v = 0; v < 5; ++v) b[v] = win[ra][v][t + H - 1 + side];
            },
            T.G.gamma, T.G.area[0], f5, fx, lwx);
        if (!finite_sum5(f5)) fx |= kFlagFlux;
        if (i <= hi0) flags |= fx;
        double lower[5];
#pragma unroll
        for (int v = 0; v < 5; ++v) {
            const double up = lane_shift_up1(f5[v]);
            // a helper lane's own difference goes unused, and where there is
            // one nothing wrote the first faces
            lower[v] = helper == 0 && t == 0 ? first[v][a - a0] : up;
        }
        if (node) {
            const SweepArgs& U = args();
            double pq[5];
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                pq[v] = win[ra][v][t + H - 1];
                if (HAS_S) s5[v] = ps[v] + s5[v];
                s5[v] = s5[v] + (f5[v] - lower[v]);
            }
            double dl = INFINITY;
            double qn[5];
            const long long nid = id + i + xo;
            stage_update_dt<TIME>(U.G, U.A, nid, pq, pq0, s5, dt_step, flags, dl, qn);
            const SweepArgs& V = args();
            write_ends<CORNERS>(V.G, V.A.qout, i, a, k, nid, qn, flags);
            dt_local = fmin(dt_local, dl);
        }
    }
    if (WAVES > 1 && raised) return;
    raise_fault(flags, W.A.flags, W.A.fault_tag, W.A.tag);
    if (W.A.reduce_dt) wave_min_atomic<SLOTS>(dt_local, W.A.dtmin);
}

template <int SCHEME, int FLUX, int TIME, bool HAS_S, int WAVES>
__global__ __launch_bounds__(kXBlock * WAVES)
__attribute__((amdgpu_waves_per_eu(SCHEME == 3 ? 2 : 3, 8))) void k_stage_yx(SweepArgs W,
                                                                             YxShape sh) {
    __shared__ YxLds<SCHEME, WAVES> lds;
    const unsigned raised = *W.A.flags;   // tested once the window is on its way
    // blocks of one XCD take consecutive numbers (x fastest), so that they
    // share the halo lines in its L2
    const unsigned chunk = gridDim.x >> 3;
    const unsigned bid = (blockIdx.x & 7u) * chunk + (blockIdx.x >> 3);
    if (bid >= sh.blocks) return;
    const unsigned bx = bid % (unsigned)sh.nx, br = bid / (unsigned)sh.nx;
    const int k = W.G.solved_lo[2] + (int)(br / (unsigned)sh.ny);
    const int wave = WAVES > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / kXBlock) : 0;
    const int a0 =
        W.G.solved_lo[1] + ((int)(br % (unsigned)sh.ny) * WAVES + wave) * sh.rows;
    const int a1 = min(a0 + sh.rows, W.G.solved_hi[1] + 1);
    const int helper = kXBlock - sh.cols;              // 1: lane 0 only evaluates a face
    const int i0 = W.G.solved_lo[0] + (int)bx * sh.cols - helper;   // lane 0's column
    stage_yx_tile<SCHEME, FLUX, TIME, HAS_S, false, kDtSlots, WAVES>(
        W, [] () -> const SweepArgs& { return sweep_args(); }, lds, i0, helper, a0, a1, k,
        bid == 0 && wave == 0, raised);
}

}  // namespace sfamd
