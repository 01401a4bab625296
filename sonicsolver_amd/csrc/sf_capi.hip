// sf_capi.hip -- host side of the C ABI declared in include/sonic_amd.h:
// device buffers, the per-stage launch sequence and the error handling.
#include "sonic_amd.h"
#include "sf_kernels.h"
#include "sf_sweep.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <limits>
#include <mutex>
#include <new>
#include <string>
#include <utility>
#include <vector>

using namespace sfamd;

namespace {

thread_local std::string g_last_error;

int fail(int code, const std::string& msg) {
    g_last_error = msg;
    return code;
}

#define SF_HIP(call)                                                              \
    do {                                                                          \
        hipError_t e_ = (call);                                                   \
        if (e_ != hipSuccess)                                                     \
            return fail(SF_E_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

}  // namespace

namespace sfamd {
// Used by the provider layer (host/sf_provider.cpp) to report through
// sf_last_error.
void set_last_error(const std::string& message) { g_last_error = message; }
}  // namespace sfamd

namespace {

// the grid's CFL accumulator and the three that k_step_1d uses in turn
constexpr size_t kDtWords = (size_t)(1 + kStepSets) * kDtSlots * kDtStride;
constexpr size_t kDtBytes = sizeof(unsigned long long) * kDtWords;
constexpr int kPinnedDts = 480;   // dt values that come back through pinned memory

}  // namespace

struct sf_grid {
    sf_grid_desc desc{};
    GridDev G{};
    hipStream_t stream = nullptr;
    double* buf[3] = {nullptr, nullptr, nullptr};
    double* S = nullptr;
    double* k[3] = {nullptr, nullptr, nullptr};
    Control* ctl = nullptr;      // device clock and fault record
    Clock* clock = nullptr;      // &ctl->clock
    Fault* fault = nullptr;      // &ctl->fault
    unsigned* flags = nullptr;   // &ctl->fault.flags
    unsigned long long* slots = nullptr;   // CFL accumulator
    // Pinned host memory (null for sf_run_static): what k_clock last wrote
    // there, followed by kPinnedDts doubles.  snapped: it is up to date once
    // the stream has been waited for.
    Control* host = nullptr;
    int snapped = 0;
    long long seq = 0;           // sequence number of the next step to begin
    // The step with sequence number base_seq starts from buffer base_cur;
    // each step moves the current state by a fixed rotation of the three
    // buffers (plan_buffers), so the buffer a later step started from
    // follows from its sequence number.
    long long base_seq = 0;
    int base_cur = 0;
    int march_seg = 0;           // nodes per march segment (0: automatic)
    int x_walk = -1;             // x sweep by lines (1), by flat tiles (0), automatic (-1)
    int cus = 256;               // compute units of the grid's device
    double* dt_hist = nullptr;
    int dt_hist_cap = 0;
    double* stage_io = nullptr;  // unique-node staging for transfers
    size_t bytes = 0;
    int cur = 0;                 // buffer holding the current state
    int ghosts_valid = 0;        // buf[cur]'s boundary is prepared as far as map_node needs it
    int stored = 0;              // buf[cur] holds all boundary nodes and ghosts (k_fill)
    int separate = 0;            // the last stage ran the separate x sweep
    int raw = 0;                 // buf[cur] is an upload whose boundary is not prepared yet
    int dtmin_valid = 0;         // the CFL accumulator holds the scan of buf[cur]
    double dtmin_cfl = 0.0;      // CFL number the folded scan used
    int step_open = 0;
    int next_stage = 0;
    int run_step = -1;           // step of a run whose steps keep the clock (StepClock), or -1
    double* run_hist = nullptr;  // its dt values go here
    int stage_in[4] = {0, 0, 0, 0}, stage_out[4] = {0, 0, 0, 0};
    double step_cfl = 0.5;       // CFL folded into the last stage's update
    int fold_cfl = 0;
    double max_dt = std::numeric_limits<double>::max();
    double limit = std::numeric_limits<double>::max();
    // kernel timing (sf_profile_*): event pairs recorded around launches
    int profiling = 0;
    std::vector<hipEvent_t> ev_pool;
    std::vector<std::pair<int, int>> ev_used;  // (kernel, index of start event)
};

namespace {

int nstages(int time) { return time == SF_TIME_EULER ? 1 : time == SF_TIME_SSPRK3 ? 3 : 4; }

int check_desc(const sf_grid_desc* d) {
    if (!d) return fail(SF_E_ARG, "sf_grid_create: null description");
    int nact = 0;
    for (int a = 0; a < 3; ++a) {
        if (d->active[a] != 0 && d->active[a] != 1)
            return fail(SF_E_ARG, "active[] entries must be 0 or 1");
        if (d->active[a]) {
            ++nact;
            if (d->n[a] < 4) return fail(SF_E_ARG, "an active axis needs at least 4 nodes");
            if (d->bc[a] < SF_BC_TRANSMISSIVE || d->bc[a] > SF_BC_NONE)
                return fail(SF_E_ARG, "unknown boundary kind");
        } else if (d->n[a] != 1) {
            return fail(SF_E_ARG, "an inactive axis must have exactly one node");
        }
        if (!(d->d[a] > 0.0) || !std::isfinite(d->d[a]))
            return fail(SF_E_ARG, "node spacing must be positive and finite");
    }
    if (nact == 0) return fail(SF_E_ARG, "at least one axis must be active");
    if (!d->active[0]) return fail(SF_E_ARG, "the x axis must be active");
    if (d->active[2] && !d->active[1])
        return fail(SF_E_ARG, "a z-active grid must also be y-active");
    if (!(d->gamma > 1.0) || !std::isfinite(d->gamma)) return fail(SF_E_ARG, "gamma must exceed 1");
    if (d->scheme < SF_SCHEME_WENO5 || d->scheme > SF_SCHEME_WENO7)
        return fail(SF_E_ARG, "unknown reconstruction scheme");
    if (d->flux < SF_FLUX_RUSANOV || d->flux > SF_FLUX_LAX_WENDROFF)
        return fail(SF_E_ARG, "unknown face flux");
    if (d->time != SF_TIME_EULER && d->time != SF_TIME_SSPRK3 && d->time != SF_TIME_RK4)
        return fail(SF_E_ARG, "unknown time recipe");
    const long long N = (long long)d->n[0] * d->n[1] * d->n[2];
    if (N > (1LL << 31)) return fail(SF_E_ARG, "grid exceeds 2^31 nodes");
    // padded nodes (ghost layers of the widest halo) index in 32 bits; no
    // grid that fits HBM with its four state buffers comes near the limit
    long long P = 1;
    for (int a = 0; a < 3; ++a) P *= a == 0 ? d->n[0] + 36 : d->active[a] ? d->n[a] + 8 : 1;
    if (P >= (1LL << 31)) return fail(SF_E_ARG, "grid exceeds 2^31 padded nodes");
    // the x sweep numbers faces in 32 bits
    if ((long long)(d->n[0] + 1) * d->n[1] * d->n[2] >= (1LL << 32) - 256)
        return fail(SF_E_ARG, "grid has 2^32 - 2^8 or more x faces");
    return 0;
}

unsigned blocks_for(long long n, int block) { return (unsigned)((n + block - 1) / block); }

// Start / stop of a timed section on the grid's stream (no-ops unless
// profiling is enabled).
int prof_start(sf_grid* g, int kernel) {
    if (!g->profiling) return -1;
    const size_t need = 2 * (g->ev_used.size() + 1);
    while (g->ev_pool.size() < need) {
        hipEvent_t e;
        if (hipEventCreate(&e) != hipSuccess) return -1;
        g->ev_pool.push_back(e);
    }
    const int idx = (int)(2 * g->ev_used.size());
    g->ev_used.push_back({kernel, idx});
    (void)hipEventRecord(g->ev_pool[idx], g->stream);
    return idx;
}

void prof_stop(sf_grid* g, int idx) {
    if (idx >= 0) (void)hipEventRecord(g->ev_pool[idx + 1], g->stream);
}

// Stores the boundary nodes and ghosts of q (k_fill).
int fill_ghosts(sf_grid* g, double* q, long long tag) {
    const GridDev& G = g->G;
    FillCount F{};
    long long n = 0;
    for (int a = 0; a < 3; ++a) {
        if (G.active[a] && (G.wrap[a] || zg_end(G, a, 0) || zg_end(G, a, 1)))
            n += 2LL * (G.g[a] + 1) * G.n[(a + 1) % 3] * G.n[(a + 2) % 3];
        F.end[a] = n;
    }
    if (n == 0) return 0;
    g->snapped = 0;
    const int ev = prof_start(g, SF_KERNEL_GHOST);
    k_fill<<<blocks_for(n, 256), 256, 0, g->stream>>>(G, q, F, g->fault, tag);
    prof_stop(g, ev);
    SF_HIP(hipGetLastError());
    return 0;
}

// Sweeps run z, y, then x: the x sweep (one face per lane) applies the
// stage update, because its register footprint is the smallest and the
// update adds to it.  The flux differences are therefore summed as
// (dz + dy) + dx rather than the reference's (dx + dy) + dz, which changes
// the last bit at most.
// The separate x sweeps read stored ghosts (`stored`: q has them); the fused
// launch reads the boundary nodes and first ghosts that a fused stage or a
// fill wrote (`closed`: q has those).
int run_sweeps(sf_grid* g, double* q, const StageArgs& A, bool stored, bool closed) {
    SweepCall c{g->G, q, g->S, A, g->stream, g->march_seg, g->cus, g->x_walk};
    auto sweep = [&](int axis, int mode) {
        switch (g->desc.scheme) {
        case SF_SCHEME_TENO5: return launch_sweep<1>(c, g->desc.flux, axis, mode);
        case SF_SCHEME_WENO3: return launch_sweep<2>(c, g->desc.flux, axis, mode);
        case SF_SCHEME_WENO7: return launch_sweep<3>(c, g->desc.flux, axis, mode);
        default: return launch_sweep<0>(c, g->desc.flux, axis, mode);
        }
    };
    auto fused = [&](const YxShape& sh) {
        switch (g->desc.scheme) {
        case SF_SCHEME_TENO5: return launch_yx<1>(c, g->desc.flux, sh);
        case SF_SCHEME_WENO3: return launch_yx<2>(c, g->desc.flux, sh);
        case SF_SCHEME_WENO7: return launch_yx<3>(c, g->desc.flux, sh);
        default: return launch_yx<0>(c, g->desc.flux, sh);
        }
    };
    const YxShape yx = yx_shape(c);
    g->separate = yx.blocks == 0;
    g->snapped = 0;
    if (g->separate ? !stored : !closed)
        if (int rc = fill_ghosts(g, q, A.tag)) return rc;
    int axes[3], na = 0;
    for (int a = 2; a >= 0; --a)
        if (g->G.active[a] && !(a == 1 && yx.blocks)) axes[na++] = a;
    for (int t = 0; t < na; ++t) {
        const bool last = t == na - 1;
        const int mode = last ? kFinal : (t == 0) ? kCopyS : kAccumS;
        const int ev = prof_start(g, SF_KERNEL_SWEEP_X + axes[t]);
        const int rc = last && yx.blocks ? fused(yx) : sweep(axes[t], mode);
        prof_stop(g, ev);
        if (rc) return fail(SF_E_STATE, "run_sweeps: no kernel for this sweep axis and mode");
    }
    SF_HIP(hipGetLastError());
    return 0;
}

int set_device(const sf_grid* g) {
    SF_HIP(hipSetDevice(g->desc.device));
    return 0;
}

int ensure_hist(sf_grid* g, int n) {
    if (n <= g->dt_hist_cap) return 0;
    if (g->dt_hist) SF_HIP(hipFree(g->dt_hist));
    g->dt_hist = nullptr;
    SF_HIP(hipMalloc(&g->dt_hist, sizeof(double) * (size_t)n));
    g->dt_hist_cap = n;
    return 0;
}

// Buffers the current state moves by in one step (plan_buffers).
int rotation(int time) { return time == SF_TIME_RK4 ? 2 : 1; }

// Tags of the launches of a step (Fault::tag): the open step's stages and
// fills, the fill that prepares or commits a step, the CFL scan before it.
long long stage_tag(const sf_grid* g, int s) { return (g->seq - 1) * 8 + s; }
long long next_tag(const sf_grid* g, int phase) { return g->seq * 8 + phase; }

// k_clock on the grid's stream; `snap` takes a snapshot for the host.
void launch_clock(sf_grid* g, double* hist, int slot, int commit, int next_dt, bool snap) {
    k_clock<<<1, kDtSlots, 0, g->stream>>>(g->ctl, g->slots, hist, slot, commit, next_dt,
                                           snap ? g->host : nullptr);
    g->snapped = snap && g->host;
}

// Wait for the grid's work and read its fault record.  With flags raised,
// every launch after the faulting one returned at entry, so the buffer that
// held the state at the start of the faulting step still holds it: it
// becomes the current state again, and the grid's clock (which no step
// committed after the fault) counts the steps before it.  Reports the
// 1-based number of the faulting step on the clock and its phase.
int check_flags(sf_grid* g, const char* where, uint32_t* flags_out = nullptr,
                long long* step_out = nullptr, int* phase_out = nullptr) {
    Control ctl{};
    if (g->host) {
        if (!g->snapped) launch_clock(g, nullptr, 0, 0, 0, true);
        SF_HIP(hipGetLastError());
        SF_HIP(hipStreamSynchronize(g->stream));
        ctl = *g->host;
    } else {
        SF_HIP(hipMemcpyAsync(&ctl, g->ctl, sizeof ctl, hipMemcpyDeviceToHost, g->stream));
        SF_HIP(hipStreamSynchronize(g->stream));
    }
    const Fault& h = ctl.fault;
    const Clock& c = ctl.clock;
    if (flags_out) *flags_out = h.flags;
    if (step_out) *step_out = h.flags ? c.steps + 1 : 0;
    if (phase_out) *phase_out = h.flags ? (int)(h.tag & 7) : -1;
    if (!h.flags) {
        g->base_seq = g->seq;
        g->base_cur = g->cur;
        return 0;
    }
    const long long seq = h.tag >> 3;
    const int phase = (int)(h.tag & 7);
    if (seq >= g->base_seq)
        g->cur = (int)((g->base_cur + (seq - g->base_seq) * rotation(g->desc.time)) % 3);
    g->base_seq = g->seq;
    g->base_cur = g->cur;
    g->step_open = 0;
    g->ghosts_valid = 0;
    g->stored = 0;
    g->dtmin_valid = 0;
    char what[32];
    if (phase < 4) std::snprintf(what, sizeof what, "stage %d", phase + 1);
    else std::snprintf(what, sizeof what, "%s", phase == kPhaseScan ? "CFL scan" : "ghost fill");
    char msg[320];
    std::snprintf(msg, sizeof msg,
                  "%s: device raised numerical fault flags 0x%x "
                  "(1 state, 2 face average, 4 TENO cutoff, 8 flux, 16 dt) in step %lld, %s; "
                  "the grid holds the state at the start of that step",
                  where, h.flags, c.steps + 1, what);
    return fail(SF_E_NUMERIC, msg);
}

// The dt limits of the steps that follow and, unless the last stage's update
// folded it in, the CFL scan of the current state.
int scan_dt(sf_grid* g, double cfl, double max_dt, double limit) {
    const bool scan = !(g->dtmin_valid && g->dtmin_cfl == cfl);
    if (scan || g->max_dt != max_dt || g->limit != limit) {
        g->max_dt = max_dt;
        g->limit = limit;
        k_set_limits<<<1, kDtSlots, 0, g->stream>>>(g->clock, g->slots, max_dt, limit, scan);
    }
    if (scan) {
        const long long N = (long long)g->G.n[0] * g->G.n[1] * g->G.n[2];
        const unsigned nb = std::min<unsigned>(blocks_for(N, 256), 8192u);
        const int ev = prof_start(g, SF_KERNEL_CFL);
        k_cfl<<<nb, 256, 0, g->stream>>>(g->G, g->buf[g->cur], cfl, g->slots, g->fault,
                                         next_tag(g, kPhaseScan));
        prof_stop(g, ev);
        g->snapped = 0;
    }
    SF_HIP(hipGetLastError());
    g->dtmin_valid = 0;
    return 0;
}

// The accumulators of a run's steps (StepClock); step s folds into set s.
unsigned long long* step_set(const sf_grid* g, int s) {
    return g->slots + (1 + s % kStepSets) * kDtSlots * kDtStride;
}

int do_stage(sf_grid* g, int s, int fold_dt) {
    const int in = g->stage_in[s], out = g->stage_out[s];
    if (s == 0 && !g->ghosts_valid) {
        if (int rc = fill_ghosts(g, g->buf[in], stage_tag(g, s))) return rc;
        g->stored = 1;
        g->raw = 0;
    }
    StageArgs A{};
    A.fault_tag = &g->fault->tag;
    A.tag = stage_tag(g, s);
    A.q0 = g->buf[g->cur];
    A.qout = g->buf[out];
    for (int i = 0; i < 3; ++i) A.k[i] = g->k[i];
    A.dt = &g->clock->dt;
    A.dtmin = g->run_step >= 0 ? step_set(g, g->run_step) : g->slots;
    A.flags = g->flags;
    A.time = g->desc.time;
    A.stage = s;
    if (g->run_step >= 0 && s == 0) {
        A.ctl = g->ctl;
        A.scan = g->run_step > 0 ? step_set(g, g->run_step - 1) : nullptr;
        A.clear = step_set(g, g->run_step + 1);
        A.dt_hist = g->run_hist;
        A.slot = g->run_step;
    }
    if (g->desc.time == SF_TIME_SSPRK3) {
        static const double base[3] = {0.0, 0.75, 1.0 / 3.0};
        static const double incr[3] = {1.0, 0.25, 2.0 / 3.0};
        A.base = base[s];
        A.incr = incr[s];
    } else if (g->desc.time == SF_TIME_RK4) {
        static const double incr[4] = {0.5, 0.5, 1.0, 0.0};
        A.incr = incr[s];
    } else {
        A.incr = 1.0;
    }
    const bool last = s == nstages(g->desc.time) - 1;
    A.reduce_dt = (last && fold_dt) ? 1 : 0;
    A.cfl = g->step_cfl;
    // a stage by the separate sweeps leaves its output's boundary as it was
    return run_sweeps(g, g->buf[in], A, s == 0 && g->stored, s == 0 || !g->separate);
}

// Stage buffers of a step.  No stage writes the buffer that holds the
// step-start state (a), so that state survives a fault in any stage; the
// step's result lands in another buffer, which becomes the current one.
void plan_buffers(sf_grid* g) {
    const int a = g->cur, b = (a + 1) % 3, c = (a + 2) % 3;
    switch (g->desc.time) {
    case SF_TIME_EULER:
        g->stage_in[0] = a; g->stage_out[0] = b;
        break;
    case SF_TIME_SSPRK3:
        g->stage_in[0] = a; g->stage_out[0] = b;
        g->stage_in[1] = b; g->stage_out[1] = c;
        g->stage_in[2] = c; g->stage_out[2] = b;
        break;
    default:
        g->stage_in[0] = a; g->stage_out[0] = b;
        g->stage_in[1] = b; g->stage_out[1] = c;
        g->stage_in[2] = c; g->stage_out[2] = b;
        g->stage_in[3] = b; g->stage_out[3] = c;
        break;
    }
}

// Grid constants of a checked description (no device work).
void set_geometry(sf_grid* g, const sf_grid_desc* desc) {
    g->desc = *desc;
    GridDev& G = g->G;
    for (int a = 0; a < 3; ++a) {
        G.n[a] = desc->n[a];
        // ghost depth = the scheme's halo (builtInConvectionRecipe,
        // SF_termRecipe.h:217-218)
        G.g[a] = desc->active[a] ? (desc->scheme == SF_SCHEME_WENO3 ? 2
                                    : desc->scheme == SF_SCHEME_WENO7 ? 4 : 3) : 0;
        G.m[a] = G.n[a] + 2 * G.g[a];
        if (a == 0) {
            // rows start on 128-byte lines: node 0 of every row sits 16
            // doubles into it (its ghosts just before), and the row length
            // is a multiple of 16, so the marches' 64-column blocks read and
            // write whole cache lines; the row holds at least one node past
            // the last ghost, so the line-walking x sweep can copy the last
            // ghost as the first of a 16-byte pair
            G.xo = 16;
            G.m[0] = (G.xo + G.n[0] + G.g[0] + 1 + 15) / 16 * 16;
        }
        G.active[a] = desc->active[a];
        G.bc[a] = desc->bc[a];
        G.d[a] = desc->d[a];
    }
    G.div_line = make_fastdiv((unsigned)G.n[0] + 1u);
    G.div_n1 = make_fastdiv((unsigned)G.n[1]);
    for (int a = 0; a < 3; ++a) {
        G.solved_lo[a] = zg_end(G, a, 0) ? 1 : 0;
        G.solved_hi[a] = G.n[a] - 1 - (zg_end(G, a, 1) ? 1 : 0);
        G.zg_lo[a] = zg_end(G, a, 0) ? 1 : 0;
        G.zg_hi[a] = zg_end(G, a, 1) ? 1 : 0;
        G.map_lo[a] = G.zg_lo[a] ? -1 : std::numeric_limits<int>::min();
        G.map_hi[a] = G.zg_hi[a] ? G.n[a] : std::numeric_limits<int>::max();
        G.wrap[a] = desc->active[a] && desc->bc[a] == SF_BC_PERIODIC ? G.n[a] : 0;
    }
    G.stride[0] = 1;
    G.stride[1] = G.m[0];
    G.stride[2] = (long long)G.m[0] * G.m[1];
    G.P = (long long)G.m[0] * G.m[1] * G.m[2];
    for (int a = 0; a < 3; ++a) G.ustride[a] = (unsigned)G.stride[a];
    G.gamma = desc->gamma;
    // Uniform Cartesian metrics exactly as the reference forms them:
    // Jac = 1/J, metric = 1/d, face cofactor = 0.5*(metric/Jac + metric/Jac),
    // area = |cofactor| (SF_mesh.cpp:320-338, SF_canonicalFace.h:87-108).
    // The metric of an inactive axis is stored as 0: its CFL term, which
    // the reference skips, then adds an exact zero.
    G.jac = 1.0 / (desc->d[0] * desc->d[1] * desc->d[2]);
    for (int a = 0; a < 3; ++a) {
        G.metric[a] = desc->active[a] ? 1.0 / desc->d[a] : 0.0;
        const double c = (1.0 / desc->d[a]) / G.jac;
        const double cof = 0.5 * (c + c);
        G.area[a] = std::sqrt(cof * cof + 0.0 * 0.0 + 0.0 * 0.0);
    }
}

int grid_free(sf_grid* g) {
    if (g->stream) (void)hipStreamSynchronize(g->stream);
    for (double* p : g->buf) if (p) (void)hipFree(p);
    for (double* p : g->k) if (p) (void)hipFree(p);
    if (g->S) (void)hipFree(g->S);
    if (g->slots) (void)hipFree(g->slots);   // and ctl, behind it
    if (g->host) (void)hipHostFree(g->host);
    if (g->dt_hist) (void)hipFree(g->dt_hist);
    if (g->stage_io) (void)hipFree(g->stage_io);
    for (hipEvent_t e : g->ev_pool) (void)hipEventDestroy(e);
    if (g->stream) (void)hipStreamDestroy(g->stream);
    delete g;
    return 0;
}

}  // namespace

extern "C" {

int sf_last_error(char* buf, size_t len) {
    if (!buf || len == 0) return SF_E_ARG;
    std::snprintf(buf, len, "%s", g_last_error.c_str());
    return 0;
}

int sf_version(int* major, int* minor) {
    if (major) *major = 0;
    if (minor) *minor = 1;
    return 0;
}

int sf_grid_create(const sf_grid_desc* desc, sf_grid** out) {
    if (!out) return fail(SF_E_ARG, "sf_grid_create: null output handle");
    *out = nullptr;
    if (int rc = check_desc(desc)) return rc;
    int ndev = 0;
    SF_HIP(hipGetDeviceCount(&ndev));
    if (desc->device < 0 || desc->device >= ndev)
        return fail(SF_E_ARG, "sf_grid_create: device ordinal out of range");
    SF_HIP(hipSetDevice(desc->device));
    sf_grid* g = new (std::nothrow) sf_grid;
    if (!g) return fail(SF_E_MEMORY, "sf_grid_create: host allocation failed");
    set_geometry(g, desc);
    const GridDev& G = g->G;
    if (hipDeviceGetAttribute(&g->cus, hipDeviceAttributeMultiprocessorCount, desc->device) !=
            hipSuccess || g->cus <= 0)
        g->cus = 256;   // MI355X's CU count; only the launch shapes depend on it
    const size_t state = sizeof(double) * 5 * (size_t)G.P;
    const size_t N = (size_t)desc->n[0] * desc->n[1] * desc->n[2];
    auto alloc = [&](double** p, size_t bytes) -> int {
        hipError_t e = hipMalloc(p, bytes);
        if (e != hipSuccess) {
            *p = nullptr;
            return fail(SF_E_MEMORY, std::string("sf_grid_create: hipMalloc of ") +
                                         std::to_string(bytes) + " bytes failed: " +
                                         hipGetErrorString(e));
        }
        g->bytes += bytes;
        return 0;
    };
    int rc = 0;
    for (int i = 0; i < 3 && !rc; ++i) rc = alloc(&g->buf[i], state);
    if (!rc) rc = alloc(&g->S, state);
    if (!rc && desc->time == SF_TIME_RK4)
        for (int i = 0; i < 3 && !rc; ++i) rc = alloc(&g->k[i], state);
    if (!rc) rc = alloc(&g->stage_io, sizeof(double) * 5 * N);
    void* ctl = nullptr;
    if (!rc && hipMalloc(&ctl, kDtBytes + sizeof(Control)) != hipSuccess)
        rc = fail(SF_E_MEMORY, "sf_grid_create: clock allocation failed");
    if (!rc) {
        g->slots = static_cast<unsigned long long*>(ctl);
        g->ctl = reinterpret_cast<Control*>(static_cast<char*>(ctl) + kDtBytes);
        g->clock = &g->ctl->clock;
        g->fault = &g->ctl->fault;
        g->flags = &g->fault->flags;
    }
    if (!rc && hipHostMalloc((void**)&g->host, sizeof(Control) + sizeof(double) * kPinnedDts,
                             hipHostMallocDefault) != hipSuccess)
        rc = fail(SF_E_MEMORY, "sf_grid_create: pinned host allocation failed");
    if (!rc && hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking) != hipSuccess)
        rc = fail(SF_E_HIP, "sf_grid_create: stream creation failed");
    if (rc) {
        grid_free(g);
        return rc;
    }
    Control c{};
    c.clock.max_dt = g->max_dt;
    c.clock.limit = g->limit;
    c.fault.tag = -1;
    std::vector<unsigned long long> init(kDtWords + sizeof c / 8, 0x7FF0000000000000ull);
    static_assert(sizeof c % 8 == 0, "copied behind the accumulators");
    std::memcpy(init.data() + kDtWords, &c, sizeof c);
    if (hipMemcpy(g->slots, init.data(), init.size() * 8, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemsetAsync(g->buf[0], 0, state, g->stream) != hipSuccess ||
        hipMemsetAsync(g->buf[1], 0, state, g->stream) != hipSuccess ||
        hipMemsetAsync(g->buf[2], 0, state, g->stream) != hipSuccess ||
        hipMemsetAsync(g->S, 0, state, g->stream) != hipSuccess) {
        grid_free(g);
        return fail(SF_E_HIP, "sf_grid_create: initialisation copy failed");
    }
    *out = g;
    return 0;
}

int sf_grid_destroy(sf_grid* g) {
    if (!g) return 0;
    set_device(g);
    return grid_free(g);
}

int sf_grid_device_bytes(const sf_grid* g, size_t* bytes) {
    if (!g || !bytes) return fail(SF_E_ARG, "sf_grid_device_bytes: null argument");
    *bytes = g->bytes;
    return 0;
}

int sf_grid_stream(sf_grid* g, void** stream) {
    if (!g || !stream) return fail(SF_E_ARG, "sf_grid_stream: null argument");
    *stream = (void*)g->stream;
    return 0;
}

// A new state starts with a clear fault record.
static int upload_from(sf_grid* g, const double* dsrc) {
    const GridDev& G = g->G;
    const long long N = (long long)G.n[0] * G.n[1] * G.n[2];
    const unsigned nb = std::min<unsigned>(blocks_for(N, 256), 65535u);
    g->snapped = 0;
    k_clear_fault<<<1, 64, 0, g->stream>>>(g->fault);
    g->base_seq = g->seq;
    g->base_cur = g->cur;
    k_pack<<<nb, 256, 0, g->stream>>>(G, dsrc, g->buf[g->cur], 1, 0);
    // ends without a condition: every state buffer's ghost layers there hold
    // the uploaded end nodes from now on
    for (int a = 0; a < 3; ++a) {
        if (!G.active[a] || G.bc[a] < SF_BC_NONE_LO) continue;
        const unsigned np = blocks_for(2LL * G.n[(a + 1) % 3] * G.n[(a + 2) % 3], 256);
        for (int b = 0; b < 3; ++b) {
            if (a == 0) k_bc_hold<0><<<np, 256, 0, g->stream>>>(G, g->buf[g->cur], g->buf[b]);
            if (a == 1) k_bc_hold<1><<<np, 256, 0, g->stream>>>(G, g->buf[g->cur], g->buf[b]);
            if (a == 2) k_bc_hold<2><<<np, 256, 0, g->stream>>>(G, g->buf[g->cur], g->buf[b]);
        }
    }
    SF_HIP(hipGetLastError());
    g->ghosts_valid = 0;
    g->stored = 0;
    g->raw = 1;
    g->dtmin_valid = 0;
    g->step_open = 0;
    return 0;
}

int sf_state_upload(sf_grid* g, const double* soa) {
    if (!g || !soa) return fail(SF_E_ARG, "sf_state_upload: null argument");
    if (int rc = set_device(g)) return rc;
    const size_t N = (size_t)g->G.n[0] * g->G.n[1] * g->G.n[2];
    SF_HIP(hipMemcpyAsync(g->stage_io, soa, sizeof(double) * 5 * N, hipMemcpyHostToDevice,
                          g->stream));
    if (int rc = upload_from(g, g->stage_io)) return rc;
    SF_HIP(hipStreamSynchronize(g->stream));
    return 0;
}

int sf_state_upload_device(sf_grid* g, const double* soa_device) {
    if (!g || !soa_device) return fail(SF_E_ARG, "sf_state_upload_device: null argument");
    if (int rc = set_device(g)) return rc;
    return upload_from(g, soa_device);
}

static int download_to(sf_grid* g, double* ddst) {
    const long long N = (long long)g->G.n[0] * g->G.n[1] * g->G.n[2];
    const unsigned nb = std::min<unsigned>(blocks_for(N, 256), 65535u);
    k_pack<<<nb, 256, 0, g->stream>>>(g->G, g->buf[g->cur], ddst, 0, !g->raw);
    SF_HIP(hipGetLastError());
    return 0;
}

int sf_state_download(sf_grid* g, double* soa) {
    if (!g || !soa) return fail(SF_E_ARG, "sf_state_download: null argument");
    if (int rc = set_device(g)) return rc;
    if (int rc = download_to(g, g->stage_io)) return rc;
    const size_t N = (size_t)g->G.n[0] * g->G.n[1] * g->G.n[2];
    SF_HIP(hipMemcpyAsync(soa, g->stage_io, sizeof(double) * 5 * N, hipMemcpyDeviceToHost,
                          g->stream));
    SF_HIP(hipStreamSynchronize(g->stream));
    return 0;
}

int sf_state_download_device(sf_grid* g, double* soa_device) {
    if (!g || !soa_device) return fail(SF_E_ARG, "sf_state_download_device: null argument");
    if (int rc = set_device(g)) return rc;
    return download_to(g, soa_device);
}

int sf_step_prepare(sf_grid* g) {
    if (!g) return fail(SF_E_ARG, "sf_step_prepare: null grid");
    if (int rc = set_device(g)) return rc;
    if (g->step_open) return fail(SF_E_STATE, "sf_step_prepare: a step is open");
    if (!g->ghosts_valid) {
        if (int rc = fill_ghosts(g, g->buf[g->cur], next_tag(g, kPhaseFill))) return rc;
        g->ghosts_valid = 1;
        g->stored = 1;
        g->raw = 0;
    }
    return 0;
}

int sf_compute_dt(sf_grid* g, double cfl, double max_dt, double limit, double* dt_out) {
    if (!g) return fail(SF_E_ARG, "sf_compute_dt: null grid");
    if (!(cfl > 0.0) || !std::isfinite(cfl)) return fail(SF_E_ARG, "sf_compute_dt: invalid CFL");
    if (!(max_dt > 0.0) || !(limit > 0.0))
        return fail(SF_E_ARG, "sf_compute_dt: limits must be positive");
    if (int rc = set_device(g)) return rc;
    if (g->step_open) return fail(SF_E_STATE, "sf_compute_dt: a step is open");
    if (int rc = scan_dt(g, cfl, max_dt, limit)) return rc;
    launch_clock(g, nullptr, 0, 0, 1, dt_out != nullptr);
    SF_HIP(hipGetLastError());
    g->step_cfl = cfl;
    if (dt_out) {
        const int rc = check_flags(g, "sf_compute_dt");
        if (g->snapped) *dt_out = g->host->clock.dt;
        return rc;
    }
    return 0;
}

int sf_set_dt(sf_grid* g, double dt) {
    if (!g) return fail(SF_E_ARG, "sf_set_dt: null grid");
    if (!(dt > 0.0) || !std::isfinite(dt)) return fail(SF_E_ARG, "sf_set_dt: invalid dt");
    if (int rc = set_device(g)) return rc;
    if (g->step_open) return fail(SF_E_STATE, "sf_set_dt: a step is open");
    g->snapped = 0;
    k_set_dt<<<1, 64, 0, g->stream>>>(g->clock, dt);
    SF_HIP(hipGetLastError());
    return 0;
}

int sf_step_begin(sf_grid* g) {
    if (!g) return fail(SF_E_ARG, "sf_step_begin: null grid");
    if (g->step_open) return fail(SF_E_STATE, "sf_step_begin: a step is already open");
    plan_buffers(g);
    ++g->seq;
    g->step_open = 1;
    g->next_stage = 0;
    return 0;
}

int sf_stage_count(const sf_grid* g, int* count) {
    if (!g || !count) return fail(SF_E_ARG, "sf_stage_count: null argument");
    *count = nstages(g->desc.time);
    return 0;
}

int sf_stage(sf_grid* g, int stage) {
    if (!g) return fail(SF_E_ARG, "sf_stage: null grid");
    if (!g->step_open || stage != g->next_stage || stage >= nstages(g->desc.time))
        return fail(SF_E_STATE, "sf_stage: stage out of order or no open step");
    if (int rc = set_device(g)) return rc;
    if (int rc = do_stage(g, stage, g->fold_cfl)) return rc;
    g->next_stage++;
    return 0;
}

// The step's result becomes the current state (the clock is the caller's).
static int commit_state(sf_grid* g) {
    g->cur = g->stage_out[nstages(g->desc.time) - 1];
    if (g->separate)
        if (int rc = fill_ghosts(g, g->buf[g->cur], (g->seq - 1) * 8 + kPhaseFill)) return rc;
    g->ghosts_valid = 1;
    g->stored = g->separate;
    g->dtmin_valid = g->fold_cfl;
    g->dtmin_cfl = g->step_cfl;
    g->step_open = 0;
    return 0;
}

int sf_step_commit(sf_grid* g) {
    if (!g) return fail(SF_E_ARG, "sf_step_commit: null grid");
    if (!g->step_open || g->next_stage != nstages(g->desc.time))
        return fail(SF_E_STATE, "sf_step_commit: stages incomplete");
    if (int rc = set_device(g)) return rc;
    if (int rc = commit_state(g)) return rc;
    launch_clock(g, nullptr, 0, 1, 0, true);
    SF_HIP(hipGetLastError());
    return 0;
}

// Whether a 1D grid's whole steps run in one launch each (k_step_1d), us per
// step against a launch per stage: WENO5/SSPRK3 10 / 29 at 1000 nodes, 16 /
// 34 at 65,000, 30 / 48 at 200,000, 121 / 141 at a million (TENO5 171 / 179);
// with WENO7 and RK4, whose blocks advance 32 nodes on 64 lanes, 16 / 42 at
// 1000, 45 / 56 at 100,000, 76 / 76 at 200,000, 304 / 273 at a million.
static bool whole_steps(const sf_grid* g) {
    const int advanced = 64 - 2 * g->G.g[0] * nstages(g->desc.time);
    return !g->G.active[1] && g->x_walk < 0 && g->G.n[0] <= (advanced > 32 ? 1 << 20 : 1 << 17);
}

// One step of a grid that takes whole steps.
static int whole_step(sf_grid* g, int s, double cfl, double* hist) {
    const int to = g->stage_out[nstages(g->desc.time) - 1];
    const Step1dArgs W{g->G, g->buf[g->cur], g->buf[to], g->ctl,
                       s ? step_set(g, s - 1) : nullptr, step_set(g, s), step_set(g, s + 1),
                       hist, s, cfl, stage_tag(g, 0)};
    const int ev = prof_start(g, SF_KERNEL_SWEEP_X);
    int rc;
    switch (g->desc.scheme) {
    case SF_SCHEME_TENO5: rc = launch_step1d<1>(W, g->desc.flux, g->desc.time, g->stream); break;
    case SF_SCHEME_WENO3: rc = launch_step1d<2>(W, g->desc.flux, g->desc.time, g->stream); break;
    case SF_SCHEME_WENO7: rc = launch_step1d<3>(W, g->desc.flux, g->desc.time, g->stream); break;
    default: rc = launch_step1d<0>(W, g->desc.flux, g->desc.time, g->stream); break;
    }
    prof_stop(g, ev);
    if (rc) return fail(SF_E_STATE, "sf_run: no kernel for this recipe");
    g->cur = to;
    g->ghosts_valid = 1;
    g->stored = 0;
    g->step_open = 0;
    return 0;
}

// queue_steps for a grid whose steps keep the clock by themselves: whole
// steps (k_step_1d) or fused stages (StepClock).
static int queue_run(sf_grid* g, int nsteps, double cfl, double max_dt, double* hist, bool whole) {
    if (int rc = sf_step_prepare(g)) return rc;
    if (int rc = scan_dt(g, cfl, max_dt, std::numeric_limits<double>::max())) return rc;
    launch_clock(g, hist, 0, 0, 1, false);
    g->step_cfl = cfl;
    g->run_hist = hist;
    int rc = 0;
    for (int s = 0; s < nsteps && !rc; ++s) {
        rc = sf_step_begin(g);
        if (rc) break;
        if (whole) {
            rc = whole_step(g, s, cfl, hist);
            continue;
        }
        g->run_step = s;
        for (int st = 0; st < nstages(g->desc.time) && !rc; ++st) rc = do_stage(g, st, 1);
        g->run_step = -1;
        if (!rc) rc = commit_state(g);
    }
    if (rc) return rc;
    k_close_run<<<1, kDtSlots, 0, g->stream>>>(g->ctl, g->slots, step_set(g, nsteps - 1),
                                               step_set(g, 0), g->host);
    g->snapped = g->host != nullptr;
    g->dtmin_valid = 1;
    g->dtmin_cfl = cfl;
    SF_HIP(hipGetLastError());
    return 0;
}

// Whether the stages of a step run the fused y / x launch, which keeps the
// clock in runs of steps.
static bool fused_stages(const sf_grid* g) {
    SweepCall c{g->G, nullptr, nullptr, StageArgs{}, g->stream, g->march_seg, g->cus, g->x_walk};
    c.A.time = g->desc.time;
    return yx_shape(c).blocks != 0;
}

// nsteps whole steps queued on the grid's stream, dt = min(CFL dt, max_dt)
// each; hist (device memory, may be null) receives the dt values.
static int queue_steps(sf_grid* g, int nsteps, double cfl, double max_dt, double* hist) {
    if (nsteps > 0 && whole_steps(g)) return queue_run(g, nsteps, cfl, max_dt, hist, true);
    if (nsteps > 0 && fused_stages(g)) return queue_run(g, nsteps, cfl, max_dt, hist, false);
    g->fold_cfl = 1;
    g->step_cfl = cfl;
    for (int s = 0; s < nsteps; ++s) {
        if (int rc = sf_step_prepare(g)) return rc;
        if (int rc = scan_dt(g, cfl, max_dt, std::numeric_limits<double>::max())) return rc;
        // one launch commits the step before and starts this one
        launch_clock(g, hist, s, s > 0, 1, false);
        if (int rc = sf_step_begin(g)) return rc;
        for (int st = 0; st < nstages(g->desc.time); ++st)
            if (int rc = sf_stage(g, st)) return rc;
        if (int rc = commit_state(g)) return rc;
    }
    if (nsteps > 0) launch_clock(g, nullptr, 0, 1, 0, true);
    SF_HIP(hipGetLastError());
    g->fold_cfl = 0;
    return 0;
}

int sf_run(sf_grid* g, int nsteps, double cfl, double max_dt, double* dt_seq) {
    if (!g) return fail(SF_E_ARG, "sf_run: null grid");
    if (nsteps < 0) return fail(SF_E_ARG, "sf_run: negative step count");
    if (!(cfl > 0.0) || !std::isfinite(cfl)) return fail(SF_E_ARG, "sf_run: invalid CFL");
    if (!(max_dt > 0.0)) return fail(SF_E_ARG, "sf_run: max_dt must be positive");
    if (g->step_open) return fail(SF_E_STATE, "sf_run: a step is open");
    if (int rc = set_device(g)) return rc;
    if (dt_seq && nsteps > 0) {
        if (int rc = ensure_hist(g, nsteps)) return rc;
    }
    if (int rc = queue_steps(g, nsteps, cfl, max_dt, dt_seq ? g->dt_hist : nullptr)) return rc;
    // the dt values come back with the status, through pinned memory where
    // they fit
    const bool pinned = dt_seq && nsteps <= kPinnedDts;
    double* const to = pinned ? reinterpret_cast<double*>(g->host + 1) : dt_seq;
    if (dt_seq && nsteps > 0)
        SF_HIP(hipMemcpyAsync(to, g->dt_hist, sizeof(double) * (size_t)nsteps,
                              hipMemcpyDeviceToHost, g->stream));
    const int rc = check_flags(g, "sf_run");
    if (pinned) std::copy(to, to + nsteps, dt_seq);
    return rc;
}

int sf_clock(sf_grid* g, double* time, long long* steps) {
    if (!g) return fail(SF_E_ARG, "sf_clock: null grid");
    if (int rc = set_device(g)) return rc;
    Clock c;
    SF_HIP(hipMemcpyAsync(&c, g->clock, sizeof c, hipMemcpyDeviceToHost, g->stream));
    SF_HIP(hipStreamSynchronize(g->stream));
    if (time) *time = c.time;
    if (steps) *steps = c.steps;
    return 0;
}

int sf_residual(sf_grid* g, double* soa_out) {
    if (!g || !soa_out) return fail(SF_E_ARG, "sf_residual: null argument");
    if (g->step_open) return fail(SF_E_STATE, "sf_residual: a step is open");
    if (int rc = set_device(g)) return rc;
    if (int rc = sf_step_prepare(g)) return rc;
    const int scratch = (g->cur + 1) % 3;
    const long long N = (long long)g->G.n[0] * g->G.n[1] * g->G.n[2];
    const unsigned nb = std::min<unsigned>(blocks_for(N, 256), 65535u);
    // Nodes that are not advanced have no residual.  Only the nodes are
    // cleared: the scratch buffer's ghosts beyond an end without a condition
    // are held for the steps that use the buffer next.
    SF_HIP(hipMemsetAsync(g->stage_io, 0, sizeof(double) * 5 * (size_t)N, g->stream));
    k_pack<<<nb, 256, 0, g->stream>>>(g->G, g->stage_io, g->buf[scratch], 1, 0);
    StageArgs A{};
    A.q0 = g->buf[g->cur];   // a valid state, though the residual-only update reads none
    A.qout = g->buf[scratch];
    A.flags = g->flags;
    A.time = 3;  // residual only
    A.dt = &g->clock->dt;
    A.dtmin = g->slots;
    A.fault_tag = &g->fault->tag;
    A.tag = next_tag(g, 0);
    if (int rc = run_sweeps(g, g->buf[g->cur], A, g->stored != 0, true)) return rc;
    k_pack<<<nb, 256, 0, g->stream>>>(g->G, g->buf[scratch], g->stage_io, 0, 0);
    SF_HIP(hipGetLastError());
    SF_HIP(hipMemcpyAsync(soa_out, g->stage_io, sizeof(double) * 5 * (size_t)N,
                          hipMemcpyDeviceToHost, g->stream));
    SF_HIP(hipStreamSynchronize(g->stream));
    return check_flags(g, "sf_residual");
}

int sf_error_flags(sf_grid* g, uint32_t* flags, int clear) {
    if (!g || !flags) return fail(SF_E_ARG, "sf_error_flags: null argument");
    if (int rc = set_device(g)) return rc;
    unsigned h = 0;
    SF_HIP(hipMemcpyAsync(&h, g->flags, sizeof h, hipMemcpyDeviceToHost, g->stream));
    SF_HIP(hipStreamSynchronize(g->stream));
    *flags = h;
    if (clear) {
        g->snapped = 0;
        k_clear_fault<<<1, 64, 0, g->stream>>>(g->fault);
        SF_HIP(hipGetLastError());
        SF_HIP(hipStreamSynchronize(g->stream));
    }
    return 0;
}

int sf_fault_check(sf_grid* g, uint32_t* flags, long long* step, int* phase) {
    if (!g) return fail(SF_E_ARG, "sf_fault_check: null grid");
    if (int rc = set_device(g)) return rc;
    return check_flags(g, "sf_fault_check", flags, step, phase);
}

int sf_grid_set_x_walk(sf_grid* g, int mode) {
    if (!g) return fail(SF_E_ARG, "sf_grid_set_x_walk: null grid");
    if (mode < -1 || mode > 1)
        return fail(SF_E_ARG, "sf_grid_set_x_walk: -1 (automatic), 0 (flat tiles) or 1 (lines)");
    g->x_walk = mode;
    return 0;
}

int sf_grid_set_march_segment(sf_grid* g, int nodes) {
    if (!g) return fail(SF_E_ARG, "sf_grid_set_march_segment: null grid");
    if (nodes != 0 && (nodes < 1 || nodes > 4096))
        return fail(SF_E_ARG, "sf_grid_set_march_segment: 0 (automatic) or 1..4096 nodes");
    g->march_seg = nodes;
    return 0;
}

int sf_profile_enable(sf_grid* g, int enable) {
    if (!g) return fail(SF_E_ARG, "sf_profile_enable: null grid");
    if (int rc = set_device(g)) return rc;
    SF_HIP(hipStreamSynchronize(g->stream));
    g->ev_used.clear();
    g->profiling = enable ? 1 : 0;
    return 0;
}

int sf_profile_read(sf_grid* g, int kernel, double* total_ms, long long* launches) {
    if (!g || kernel < 0 || kernel >= SF_KERNEL_COUNT)
        return fail(SF_E_ARG, "sf_profile_read: invalid argument");
    if (int rc = set_device(g)) return rc;
    SF_HIP(hipStreamSynchronize(g->stream));
    double sum = 0.0;
    long long n = 0;
    for (const auto& u : g->ev_used) {
        if (u.first != kernel) continue;
        float ms = 0.0f;
        SF_HIP(hipEventElapsedTime(&ms, g->ev_pool[u.second], g->ev_pool[u.second + 1]));
        sum += ms;
        ++n;
    }
    if (total_ms) *total_ms = sum;
    if (launches) *launches = n;
    return 0;
}

int sf_synchronize(sf_grid* g) {
    if (!g) return fail(SF_E_ARG, "sf_synchronize: null grid");
    if (int rc = set_device(g)) return rc;
    SF_HIP(hipStreamSynchronize(g->stream));
    return 0;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// A whole run that allocates nothing (sf_run_static): the grid's buffers,
// clock and fault record live in one file-scope device array per GPU.
// ---------------------------------------------------------------------------
namespace {

constexpr size_t kStaticBytes = size_t(64) << 20;
__device__ __align__(256) unsigned char scratch[kStaticBytes];
__device__ __align__(128) unsigned long long scratch_slots[kDtWords];

// Device address of `scratch` on each device (its name is only a host-side
// stand-in), taken once per device with that device current.
constexpr int kMaxDevices = 64;
unsigned char* g_scratch[kMaxDevices] = {};
unsigned long long* g_scratch_slots[kMaxDevices] = {};
std::mutex g_scratch_mutex;

int static_scratch(int device, unsigned char** out, unsigned long long** slots) {
    if (device < 0 || device >= kMaxDevices)
        return fail(SF_E_ARG, "sf_run_static: device ordinal out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch[device]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(SF_E_HIP, std::string("sf_run_static: hipGetSymbolAddress: ") +
                                      hipGetErrorString(e));
        void* ps = nullptr;
        const hipError_t es = hipGetSymbolAddress(&ps, HIP_SYMBOL(scratch_slots));
        if (es != hipSuccess || !ps)
            return fail(SF_E_HIP, std::string("sf_run_static: hipGetSymbolAddress: ") +
                                      hipGetErrorString(es));
        g_scratch[device] = static_cast<unsigned char*>(p);
        g_scratch_slots[device] = static_cast<unsigned long long*>(ps);
    }
    *out = g_scratch[device];
    *slots = g_scratch_slots[device];
    return 0;
}

size_t round256(size_t bytes) { return (bytes + 255) & ~size_t(255); }

__global__ __launch_bounds__(256) void k_zero(double* __restrict__ p, long long n) {
    for (long long u = blockIdx.x * (long long)blockDim.x + threadIdx.x; u < n;
         u += (long long)gridDim.x * blockDim.x)
        p[u] = 0.0;
}

__global__ __launch_bounds__(kDtSlots) void k_init_clock(Clock* c, unsigned long long* slots) {
    for (int s = 0; s <= kStepSets; ++s)
        slots[(s * kDtSlots + threadIdx.x) * kDtStride] = 0x7FF0000000000000ull;
    if (threadIdx.x == 0) {
        c->dt = 0.0;
        c->time = 0.0;
        c->steps = 0;
        c->max_dt = std::numeric_limits<double>::max();
        c->limit = std::numeric_limits<double>::max();
    }
}

}  // namespace

extern "C" int sf_run_static(const sf_grid_desc* desc, double* soa_device, int nsteps,
                             double cfl, double max_dt, double* dt_seq_device, void* stream,
                             size_t* scratch_bytes) {
    if (!soa_device) return fail(SF_E_ARG, "sf_run_static: null state");
    if (nsteps < 0) return fail(SF_E_ARG, "sf_run_static: negative step count");
    if (!(cfl > 0.0) || !std::isfinite(cfl)) return fail(SF_E_ARG, "sf_run_static: invalid CFL");
    if (!(max_dt > 0.0)) return fail(SF_E_ARG, "sf_run_static: max_dt must be positive");
    if (int rc = check_desc(desc)) return rc;
    int ndev = 0;
    SF_HIP(hipGetDeviceCount(&ndev));
    if (desc->device < 0 || desc->device >= ndev)
        return fail(SF_E_ARG, "sf_run_static: device ordinal out of range");
    sf_grid g;
    set_geometry(&g, desc);
    if (hipDeviceGetAttribute(&g.cus, hipDeviceAttributeMultiprocessorCount, desc->device) !=
            hipSuccess || g.cus <= 0)
        g.cus = 256;
    // scratch layout: clock and fault record (512 bytes), then the state buffers, the flux
    // accumulator and (RK4) the three stage residuals
    const size_t state = round256(sizeof(double) * 5 * (size_t)g.G.P);
    const int nbuf = desc->time == SF_TIME_RK4 ? 7 : 4;
    const size_t head = 512;
    const size_t need = head + state * nbuf;
    if (scratch_bytes) *scratch_bytes = need;
    if (need > kStaticBytes) {
        char msg[256];
        std::snprintf(msg, sizeof msg,
                      "sf_run_static: the grid needs %zu bytes of device scratch, more than "
                      "the %zu bytes the library holds per device; use sf_grid_create",
                      need, kStaticBytes);
        return fail(SF_E_ARG, msg);
    }
    SF_HIP(hipSetDevice(desc->device));
    unsigned char* base = nullptr;
    if (int rc = static_scratch(desc->device, &base, &g.slots)) return rc;
    g.stream = static_cast<hipStream_t>(stream);
    static_assert(sizeof(Control) <= 512, "the head of the scratch layout");
    g.ctl = reinterpret_cast<Control*>(base);
    g.clock = &g.ctl->clock;
    g.fault = &g.ctl->fault;
    g.flags = &g.fault->flags;
    double* bufs[7];
    for (int i = 0; i < nbuf; ++i) bufs[i] = reinterpret_cast<double*>(base + head + state * i);
    for (int i = 0; i < 3; ++i) g.buf[i] = bufs[i];
    g.S = bufs[3];
    if (nbuf == 7)
        for (int i = 0; i < 3; ++i) g.k[i] = bufs[4 + i];
    // Every call on this device shares the array and finds the last call's
    // contents: the clock, the fault record and the buffers start cleared.
    k_init_clock<<<1, kDtSlots, 0, g.stream>>>(g.clock, g.slots);
    k_clear_fault<<<1, 64, 0, g.stream>>>(g.fault);
    const long long words = (long long)(state * nbuf / sizeof(double));
    k_zero<<<std::min<unsigned>(blocks_for(words, 256), 4096u), 256, 0, g.stream>>>(bufs[0], words);
    SF_HIP(hipGetLastError());
    if (int rc = upload_from(&g, soa_device)) return rc;
    if (int rc = queue_steps(&g, nsteps, cfl, max_dt, nsteps > 0 ? dt_seq_device : nullptr))
        return rc;
    const int status = check_flags(&g, "sf_run_static");
    if (status != 0 && status != SF_E_NUMERIC) return status;
    if (int rc = download_to(&g, soa_device)) return rc;
    SF_HIP(hipStreamSynchronize(g.stream));
    return status;
}
