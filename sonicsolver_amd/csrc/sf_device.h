// sf_device.h -- device-side pieces shared by the grid kernels and the
// batched ones: grid descriptor, stage-update arithmetic, validation flags,
// CFL folding and the energies of the boundary closure.
#pragma once

#include "sf_face.h"

namespace sfamd {

// Unsigned 32-bit division by a divisor fixed for a whole launch, as a
// multiply-high, an add and a shift (Granlund and Montgomery, "Division by
// invariant integers using multiplication", PLDI 1994, section 4): with
// l = ceil(log2 d) and m = floor(2^32 (2^l - d) / d) + 1,
// floor(x / d) = (umulhi(x, m) + x) >> l for every x < 2^32 (the sum is
// formed in 64 bits).  The host forms (m, l) with make_fastdiv.
struct FastDiv {
    unsigned m;
    unsigned l;
};

inline FastDiv make_fastdiv(unsigned d) {
    unsigned l = 0;
    while (l < 32 && (1ull << l) < d) ++l;
    FastDiv f;
    f.m = (unsigned)((((1ull << l) - d) << 32) / d + 1);
    f.l = l;
    return f;
}

__device__ __forceinline__ unsigned fast_div(unsigned x, FastDiv f) {
    const unsigned t = __umulhi(x, f.m);
    return (unsigned)(((unsigned long long)t + x) >> f.l);
}

struct GridDev {
    int n[3];
    int g[3];
    int m[3];
    int xo;             // position of node i = 0 in its row (a multiple of 16)
    long long P;        // padded nodes per variable (below 2^31)
    long long stride[3];
    unsigned ustride[3];  // the strides in 32 bits, for node_index
    int active[3];
    int bc[3];          // SF_BC_* kind of each axis
    double jac, area[3], gamma;
    double metric[3];   // 1 / spacing on active axes, 0 on inactive ones
    double d[3];        // node spacing (the Lax-Wendroff flux's face spacing)
    // Where the value of a ghost is read from, per axis (map_node): beyond a
    // zeroGradient end from its first ghost layer, which every layer equals,
    // beyond a periodic one from the node a period away; an end without a
    // condition keeps its stored ghosts.
    int map_lo[3], map_hi[3], wrap[3];
    int zg_lo[3], zg_hi[3];   // 1 where the end carries zeroGradient
    // Nodes the stage advances along each axis: solved_lo[a] .. solved_hi[a]
    // (a zeroGradient end's node is excluded; see solved_node).
    int solved_lo[3], solved_hi[3];
    // The x sweep's face -> (line, node) and line -> (j, k) divisions:
    // by n0 + 1 faces per line and by n1 lines per z plane.
    FastDiv div_line, div_n1;
};

enum { kCopyS = 0, kAccumS = 1, kFinal = 2 };

// Stage update parameters (Time::Explicit, SF_explicit.cpp:193-238).
struct StageArgs {
    const double* q0;        // step-start state (SSPRK3, RK4)
    double* qout;            // new state
    double* k[3];            // RK4 stage residuals k1..k3
    const double* dt;        // device scalar: dt of this step
    unsigned long long* dtmin;  // CFL accumulator (kDtSlots slots)
    unsigned* flags;
    double base, incr;       // SSPRK3 base / increment weights
    double cfl;
    int time;                // 0 Euler, 1 SSPRK3, 2 RK4
    int stage;
    int reduce_dt;           // fold the next step's CFL scan into this update
    long long* fault_tag;    // where the first fault is recorded (may be null)
    long long tag;           // this launch's tag (step sequence * 8 + phase)
    // Steps that keep the clock by themselves (StepClock): the grid's control
    // block and the CFL accumulator to clear, for the first stage of a step;
    // scan, where that stage has to form dt and commit the step before.
    struct Control* ctl;
    const unsigned long long* scan;   // accumulator holding this step's dt
    unsigned long long* clear;
    double* dt_hist;         // may be null
    int slot;
};

// Fault record of a grid: the flags raised since they were last cleared,
// and the tag of the launch that raised the first of them: step sequence
// number * 8 + phase (0..3 the stage, its ghost fill included; 6 the ghost
// fill at the start or commit of the step; 7 the CFL scan before it).
// Once flags are raised, every later launch of a stage, fill or clock
// kernel returns at entry, so the state at the start of the faulting step
// stays as it was.
struct Fault {
    unsigned flags;
    unsigned stages;   // k_step_1d: the flags raised by stage s at bits 8 s
    long long tag;
    unsigned before;   // the flags as the last clock launch found them
    unsigned unused;
};
enum { kPhaseFill = 6, kPhaseScan = 7 };

// Padded index of node (i, j, k); the host keeps P below 2^31, so it is
// formed in 32-bit arithmetic.
__device__ __forceinline__ long long node_index(const GridDev& G, int i, int j, int k) {
    return (long long)((unsigned)(k + G.g[2]) * G.ustride[2] + (unsigned)(j + G.g[1]) * G.ustride[1]
                       + (unsigned)(i + G.xo));
}

// Boundary kind per axis (SF_BC_*): 0 zeroGradient on both ends,
// 1 periodic, 2 / 3 / 4 no condition on the lower / upper / both ends (the
// other end zeroGradient).  zg_end: the end (side 0 lower, 1 upper) carries
// zeroGradient.
__host__ __device__ __forceinline__ bool zg_end(const GridDev& G, int d, int side) {
    const int b = G.bc[d];
    return G.active[d] && (b == 0 || (b == 2 && side == 1) || (b == 3 && side == 0));
}

// A node is advanced unless it lies on a zeroGradient end, which the
// boundary applicator marks as a solver-boundary point
// (SF_applicator.h:162-187); an end without a condition is not marked.
// The host folds that rule into the per-axis ranges solved_lo / solved_hi.
__device__ __forceinline__ bool solved_node(const GridDev& G, int i, int j, int k) {
    return i >= G.solved_lo[0] && i <= G.solved_hi[0] && j >= G.solved_lo[1] &&
           j <= G.solved_hi[1] && k >= G.solved_lo[2] && k <= G.solved_hi[2];
}

// Local CFL step of RusanovEOS::deltaT (SF_rusanovEOS.cpp:110-147).  The
// metric of an inactive axis is zero, so its term adds an exact zero.
__device__ __forceinline__ double local_dt(const GridDev& G, const double q[5], double cfl,
                                           unsigned& flags) {
    const Closed s = close_state(q, G.gamma);
    const double c = s.c();
    double spectral = 0.0;
#pragma unroll
    for (int d = 0; d < 3; ++d)
        spectral += fma(c, G.metric[d], fabs(s.u[d] * G.metric[d]));
    if (!(spectral > 0.0) || !isfinite(spectral)) flags |= kFlagDt;
    return cfl / spectral;
}

// A 64-bit value moved across lanes by one DPP control (two 32-bit moves);
// lanes whose row ROWS leaves out keep their own value.
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ unsigned long long dpp_u64(unsigned long long v) {
    const int lo = (int)(unsigned)v, hi = (int)(unsigned)(v >> 32);
    const unsigned l = (unsigned)__builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWS, 0xf, false);
    const unsigned h = (unsigned)__builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWS, 0xf, false);
    return ((unsigned long long)h << 32) | l;
}

template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ unsigned long long dpp_min_step(unsigned long long b) {
    const unsigned long long o = dpp_u64<CTRL, ROWS>(b);
    return o < b ? o : b;
}

// Minimum of b over the 64 lanes of a wave, all of them active, by DPP
// moves (no LDS): lane pairs and quads by quad permutations, 8- and
// 16-lane rows by the half-row and row mirrors, then row 0 into row 1 and
// row 2 into row 3 by the row-15 broadcast and rows 0-1 into rows 2-3 by
// the row-31 broadcast, which leaves the minimum in lane 63.
__device__ __forceinline__ unsigned long long wave_min_bits(unsigned long long b) {
    b = dpp_min_step<0xB1>(b);         // quad_perm [1,0,3,2]
    b = dpp_min_step<0x4E>(b);         // quad_perm [2,3,0,1]
    b = dpp_min_step<0x141>(b);        // row_half_mirror
    b = dpp_min_step<0x140>(b);        // row_mirror
    b = dpp_min_step<0x142, 0xa>(b);   // row_bcast:15 into rows 1 and 3
    b = dpp_min_step<0x143, 0xc>(b);   // row_bcast:31 into rows 2 and 3
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, 63);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), 63);
    return ((unsigned long long)hi << 32) | lo;
}

// CFL accumulator of a grid: the minimum is kept in kDtSlots partial minima
// (bits of positive doubles), one per 128-byte line.  Atomics on one address
// pass one by one, about 12 ns each: with a single word the scan of 853^2
// took 133 us for its 11,368 waves, of 2048^2 380, and the blocks of a stage
// that end together queued likewise.
constexpr int kDtSlots = 64, kDtStride = 16;

// Wave-wide minimum of a positive double into the accumulator (one atomic per
// wave; every lane of the wave calls it).  Positive doubles order like their
// bit patterns; a lane without a value contributes +infinity.
template <int SLOTS = kDtSlots>
__device__ __forceinline__ void wave_min_atomic(double v, unsigned long long* slots) {
    const unsigned long long b = wave_min_bits(
        (v > 0.0 && isfinite(v)) ? (unsigned long long)__double_as_longlong(v)
                                 : 0x7FF0000000000000ull);
    if ((threadIdx.x & 63) == 0 && b != 0x7FF0000000000000ull)
        atomicMin(slots + (blockIdx.x % SLOTS) * kDtStride, b);
}

// Whether all five values are finite, from their sum: a NaN or an infinity
// among them makes the sum non-finite, and finite values make it finite
// unless it overflows, which only states already far outside the range of
// this path's data could do.
__device__ __forceinline__ bool finite_sum5(const double f[5]) {
    return isfinite(((f[0] + f[1]) + (f[2] + f[3])) + f[4]);
}

// The same test without that exception: the sum of the eighths does not
// overflow.
__device__ __forceinline__ bool finite5(const double f[5]) {
    constexpr double e = 0.125;
    return isfinite(fma(e, f[4], fma(e, f[3], e * f[2]) + fma(e, f[1], e * f[0])));
}

// Raises flags f, recording the lowest tag (-1: none) before they are seen.
__device__ __forceinline__ void raise_fault(unsigned f, unsigned* flags, long long* tag_out,
                                            long long tag) {
    if (!f) return;
    if (tag_out) {
        atomicMin((unsigned long long*)tag_out, (unsigned long long)tag);
        __threadfence();
    }
    atomicOr(flags, f);
}

// The coordinate along axis a whose stored value stands for coordinate c, a
// node or ghost within the halo.
__host__ __device__ __forceinline__ int map_node(const GridDev& G, int a, int c) {
    c = min(max(c, G.map_lo[a]), G.map_hi[a]);
    c += c < 0 ? G.wrap[a] : 0;
    return c - (c >= G.n[a] ? G.wrap[a] : 0);
}

// Energies of a zeroGradient end whose inner neighbour holds q: density and
// momentum are the neighbour's, the boundary node's energy is rebuilt from
// the neighbour's pressure and the ghosts' from the boundary node's
// (SF_zeroGradient.cpp:88-130, SF_thermodynamicClosure.cpp:219-281), in the
// reference's own order of operations: both equal q[4] up to rounding, and a
// run that amplifies rounding at an outflow end follows the reference only
// if that is rounded as there.  ok: both pressures are positive.
struct EndEnergy {
    double node, ghost;
    bool ok;
};

__device__ __forceinline__ EndEnergy end_energy(const double q[5], double gamma) {
    const double r = q[0], inv = frcp(r);
    const double u = q[1] * inv, v = q[2] * inv, w = q[3] * inv;
    const double kin = 0.5 * r * (u * u + v * v + w * w);
    const double kinetic = 0.5 * inv * (q[1] * q[1] + q[2] * q[2] + q[3] * q[3]);
    const double d = (gamma - 1.0) * r, rd = frcp(d);
    const auto rebuilt = [&](double p) {
        const double x = p * rd;
        return r * fma(fma(-d, x, p), rd, x) + kinetic;
    };
    const double ps = d * ((q[4] - kin) * inv);
    EndEnergy e;
    e.node = rebuilt(ps);
    const double pb = d * ((e.node - kin) * inv);
    e.ghost = rebuilt(pb);
    e.ok = ps > 0.0 && pb > 0.0;
    return e;
}

// validateEquationState (SF_equationState.h:25-57): rho, p > 0, finite (p has
// the sign of the internal energy; with the refined reciprocal of the
// density instead of a division, that sign can differ only where the internal
// energy is within an ulp of the kinetic energy).
__device__ __forceinline__ void check_state(const double q[5], unsigned& flags) {
    const double ke = 0.5 * dot3(q + 1, q + 1);
    const double eint = fma(-ke, frcp(q[0]), q[4]);
    if (!(q[0] > 0.0) || !(eint > 0.0) || !isfinite(eint)) flags |= kFlagState;
}

// Stage update of one node from its current value qc and (SSPRK3 after
// the first stage, RK4) its step-start value q0v; S is the accumulated flux
// difference and dt the step's dt (*A.dt, which no kernel of a stage
// changes, so a sweep reads it once).  TIME fixes the time recipe (A.time) at
// compile time; -1 reads it from A.
template <int TIME = -1>
__device__ __forceinline__ void stage_update_dt(const GridDev& G, const StageArgs& A, long long id,
                                                const double qc[5], const double q0v[5],
                                                const double S[5], double dt, unsigned& flags,
                                                double& dt_local, double qn[5]) {
    const int time = TIME >= 0 ? TIME : A.time;
    if (time == 3) {  // residual only (diagnostics)
#pragma unroll
        for (int v = 0; v < 5; ++v) A.qout[v * G.P + id] = G.jac * S[v];
        return;
    }
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        const double R = G.jac * S[v];
        if (time == 1) {
            const double euler = fma(-dt, R, qc[v]);
            qn[v] = fma(A.incr, euler, A.base * q0v[v]);   // base = 0 in stage 1
        } else if (time == 0) {
            qn[v] = fma(-dt, R, qc[v]);
        } else if (A.stage < 3) {
            A.k[A.stage][v * G.P + id] = R;
            qn[v] = fma(-(A.incr * dt), R, q0v[v]);
        } else {
            const double sum = fma(2.0, A.k[2][v * G.P + id],
                                   fma(2.0, A.k[1][v * G.P + id], A.k[0][v * G.P + id])) + R;
            qn[v] = fma(-(dt / 6.0), sum, q0v[v]);
        }
        A.qout[v * G.P + id] = qn[v];
    }
    check_state(qn, flags);
    if (A.reduce_dt) dt_local = local_dt(G, qn, A.cfl, flags);
}

// Device clock: dt of the step, physical time, step count and the dt limits.
struct Clock {
    double dt;
    double time;
    long long steps;
    double max_dt;
    double limit;
};

// What the host reads back: the clock and the fault record.
struct Control {
    Clock clock;
    Fault fault;
};

// The dt of a stage's step.  In a run of steps the first stage of each keeps
// the clock: every wave forms dt from the accumulator that the step before
// folded into, and the wave that calls commit() commits that step, stores dt
// for the stages after it and clears the accumulator of the step after (three
// are used in turn, so none is cleared or folded into while it is read).
// With a clock launch between the steps each took 1.7 us longer on 193 x 97
// (28.0 us now), 2.1 on 853^2 (147) and 3.4 on 64^3 (125).
// Constructed early, so that the loads are under way while the stencil is
// fetched; get() waits for them.  Every lane of the wave takes part.
struct StepClock {
    unsigned long long bits;
    double dt, max_dt, limit;
    __device__ __forceinline__ explicit StepClock(const StageArgs& A) {
        dt = *A.dt;
        if (A.scan) {
            bits = A.scan[(threadIdx.x & 63) * kDtStride];
            max_dt = A.ctl->clock.max_dt;
            limit = A.ctl->clock.limit;
        }
    }
    __device__ __forceinline__ double get(const StageArgs& A) const {
        if (!A.scan) return dt;
        const double d = __longlong_as_double((long long)wave_min_bits(bits));
        return fmin(fmin(d, max_dt), limit);
    }
    __device__ __forceinline__ void commit(const StageArgs& A, double dt_step) const {
        if (!A.clear) return;
        const int t = threadIdx.x & 63;
        A.clear[t * kDtStride] = 0x7FF0000000000000ull;
        if (!A.scan || t) return;
        // Not after a fault of an earlier step.  One that another block
        // raises in this launch does not undo the step before.
        const Fault& f = A.ctl->fault;
        if (__hip_atomic_load(&f.flags, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) &&
            (__hip_atomic_load(&f.tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >> 3) <
                (A.tag >> 3))
            return;
        Clock& c = A.ctl->clock;
        c.time += c.dt;
        c.steps += 1;
        c.dt = dt_step;
        if (A.dt_hist) A.dt_hist[A.slot] = dt_step;
    }
};

}  // namespace sfamd
