// sf_batch.hip -- batched solves of independent 1D / 2D problems of uneven
// size.  One device arena holds every admitted problem's padded SoA state;
// a stage kernel walks a table of tiles, so one launch advances all problems
// by one RK stage (two where 1D and 2D problems share the batch); each
// problem keeps its own CFL dt and clock, and its result does not depend on
// which other problems share the batch (no cross-problem arithmetic; the
// per-problem dt is a minimum, which does not depend on the order of the
// atomics).  The launches of a few steps can be captured in a hipGraph and
// replayed while the set of problems is unchanged.
//
// Boundaries are transmissive (the reference's zeroGradient sets, applied
// axis by axis as Boundary::Applicator::apply does,
// solver/boundary/SF_applicator.h:51-83), written in place by the stage that
// advances the nodes next to them (write_ends); the time recipe is SSPRK3
// (SF_builtinProviders.cpp:98-121).  Layout of problem p in the arena:
// q[v*P + off_p + (j+gy)*m0 + i+3] with m0 = nx + 6, gy = 3 for a 2D
// problem and 0 for a 1D one.
#include "sonic_amd.h"
#include "sf_batch_copy.h"
#include "sf_batch_stage.h"
#include "sf_sweep.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <limits>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <vector>

namespace sfamd {
void set_last_error(const std::string& message);

struct BatchDev {
    const ItemArgs* items;
    const int* active;   // admitted slots
    int nactive;
    double* dt;
    unsigned long long* dtmin;   // kItemDtSlots partial minima per slot
    double* time;
    long long* steps;
    const long long* target;  // a problem is live while steps < target ...
    unsigned* flags;          // ... and raised no fault flags (per problem)
    int* live;                // liveness fixed for the current step
};

constexpr int kItemDtWords = kItemDtSlots * kDtStride;

// The problems admitted since the last step (blockIdx.x = list entry,
// blockIdx.y splits the nodes): their ends are written and their CFL scan
// (RusanovEOS::deltaT, SF_rusanovEOS.cpp:110-147) goes to dtmin.
__global__ __launch_bounds__(256) void k_batch_prepare(BatchDev B, const int* __restrict__ list) {
    const int slot = list[blockIdx.x];
    const SweepArgs& W = B.items[slot].stage[0];
    const GridDev& G = W.G;
    double* const q = const_cast<double*>(W.q);
    const int nx = G.solved_hi[0] - G.solved_lo[0] + 1;
    const long long N = (long long)nx * (G.solved_hi[1] - G.solved_lo[1] + 1);
    unsigned flags = 0;
    double best = INFINITY;
    for (long long u = blockIdx.y * (long long)blockDim.x + threadIdx.x; u < N;
         u += (long long)gridDim.y * blockDim.x) {
        const int i = G.solved_lo[0] + (int)(u % nx), j = G.solved_lo[1] + (int)(u / nx);
        const long long id = node_index(G, i, j, 0);
        double qq[5];
#pragma unroll
        for (int v = 0; v < 5; ++v) qq[v] = q[v * G.P + id];
        best = fmin(best, local_dt(G, qq, W.A.cfl, flags));
        write_ends<true>(G, q, i, j, 0, id, qq, flags);
    }
    if (flags) atomicOr(&B.flags[slot], flags);
    const unsigned long long b = wave_min_bits(
        (best > 0.0 && isfinite(best)) ? (unsigned long long)__double_as_longlong(best)
                                       : 0x7FF0000000000000ull);
    if ((threadIdx.x & 63) == 0 && b != 0x7FF0000000000000ull)
        atomicMin(B.dtmin + (long long)slot * kItemDtWords + (blockIdx.y % kItemDtSlots) * kDtStride,
                  b);
}

// The clock between two steps: commits the step before (live says which
// problems took one; a problem that faulted in it is not counted) and, with
// `next`, starts the following one: its liveness is fixed, so that every
// wave of every kernel of the step takes the same decision for a problem
// even while another block raises its flags, dt is the folded CFL minimum,
// and the accumulator is cleared for the fold of the step's last stage.  A
// problem that faults during a step finishes that step's stages on its own
// nodes and is frozen from the next step on.
__global__ void k_batch_clock(BatchDev B, int next) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= B.nactive) return;
    const int slot = B.active[k];
    const bool sound = B.flags[slot] == 0;
    long long steps = B.steps[slot];
    if (B.live[slot] && sound) {
        B.time[slot] += B.dt[slot];
        B.steps[slot] = ++steps;
    }
    const bool live = next && sound && steps < B.target[slot];
    B.live[slot] = live ? 1 : 0;
    if (!live) return;
    unsigned long long* const m = B.dtmin + (long long)slot * kItemDtWords;
    unsigned long long b = m[0];
#pragma unroll
    for (int s = 1; s < kItemDtSlots; ++s) b = min(b, m[s * kDtStride]);
#pragma unroll
    for (int s = 0; s < kItemDtSlots; ++s) m[s * kDtStride] = 0x7FF0000000000000ull;
    B.dt[slot] = __longlong_as_double((long long)b);
}

__global__ void k_batch_reset(BatchDev B, const int* __restrict__ list, int n) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int slot = list[k];
#pragma unroll
    for (int s = 0; s < kItemDtSlots; ++s)
        B.dtmin[(long long)slot * kItemDtWords + s * kDtStride] = 0x7FF0000000000000ull;
    B.time[slot] = 0.0;
    B.steps[slot] = 0;
    B.dt[slot] = 0.0;
    B.flags[slot] = 0;
    B.live[slot] = 0;
}

// A problem's arguments as a kernel's first argument, read in place.
__device__ __forceinline__ const ItemArgs& item_kernarg() {
    return *(const ItemArgs*)(const __attribute__((address_space(4))) ItemArgs*)
        __builtin_amdgcn_kernarg_segment_ptr();
}

// Admission: nodes u0 .. u0+cnt-1 of a problem from pinned host memory
// (src[v*cnt + u-u0]) into its padded block, and its arguments and step limit
// into their tables.
__global__ __launch_bounds__(256) void k_batch_admit(ItemArgs, ItemArgs* __restrict__ item,
                                                     long long* __restrict__ target,
                                                     long long limit,
                                                     const double* __restrict__ src,
                                                     unsigned u0, unsigned cnt) {
    const ItemArgs& args = item_kernarg();
    if (blockIdx.x == 0) {
        constexpr unsigned words = sizeof(ItemArgs) / 8;
        for (unsigned w = threadIdx.x; w < words; w += blockDim.x)
            ((unsigned long long*)item)[w] = ((const unsigned long long*)&args)[w];
        if (threadIdx.x == 0) *target = limit;
    }
    const GridDev& G = args.stage[0].G;
    double* const q = const_cast<double*>(args.stage[0].q);
    for (unsigned u = blockIdx.x * blockDim.x + threadIdx.x; u < cnt; u += gridDim.x * blockDim.x) {
        const unsigned at = u0 + u, n0 = (unsigned)G.n[0];
        const long long id = node_index(G, (int)(at % n0), (int)(at / n0), 0);
#pragma unroll
        for (int v = 0; v < 5; ++v) q[v * G.P + id] = src[(size_t)v * cnt + u];
    }
}

// Nodes u0 .. u0+cnt-1 of a problem's state to pinned host memory
// (dst[v*cnt + u-u0], then its clock time where `time` is given).
__global__ __launch_bounds__(256) void k_batch_pack(const ItemArgs* __restrict__ item,
                                                    double* __restrict__ dst, unsigned u0,
                                                    unsigned cnt, const double* __restrict__ time) {
    const GridDev& G = item->stage[0].G;
    const double* const q = item->stage[0].q;
    if (time && blockIdx.x == 0 && threadIdx.x == 0) dst[5 * (size_t)cnt] = *time;
    for (unsigned u = blockIdx.x * blockDim.x + threadIdx.x; u < cnt; u += gridDim.x * blockDim.x) {
        const unsigned at = u0 + u, n0 = (unsigned)G.n[0];
        const long long id = node_index(G, (int)(at % n0), (int)(at / n0), 0);
#pragma unroll
        for (int v = 0; v < 5; ++v) dst[(size_t)v * cnt + u] = q[v * G.P + id];
    }
}

}  // namespace sfamd

using namespace sfamd;

namespace {

int bfail(int code, const std::string& msg) {
    set_last_error(msg);
    return code;
}

#define SF_BHIP(call)                                                                     \
    do {                                                                                  \
        hipError_t e_ = (call);                                                           \
        if (e_ != hipSuccess)                                                             \
            return bfail(SF_E_HIP, std::string(#call) + ": " + hipGetErrorString(e_));    \
    } while (0)

long long padded_nodes(const sf_batch_item& it) {
    const long long m0 = it.n[0] + 6;
    const long long m1 = it.n[1] > 1 ? it.n[1] + 6 : 1;
    return m0 * m1;
}

}  // namespace

constexpr int kPinChunks = 4;
constexpr size_t kPinBytes = 2u << 20;                       // of a chunk
constexpr long long kPinNodes = (long long)(kPinBytes / (5 * sizeof(double)));

struct sf_batch {
    // placement of a problem in the arena
    struct Item {
        long long off = 0;      // start of its padded block
        int n0 = 0, n1 = 0, m0 = 0, gy = 0;
        int scheme = 0, flux = 0;
    };
    int device = 0;
    int cus = 256;
    double gamma = 1.4;
    long long capacity = 0;     // padded nodes per variable
    int item_capacity = 0;
    hipStream_t stream = nullptr;
    hipStream_t copy_stream = nullptr;   // copy-out of finished problems
    hipEvent_t copy_after = nullptr;     // orders copy-outs after the compute stream
    double* buf[3] = {nullptr, nullptr, nullptr};
    // Pinned host memory that kernels read admitted states from and write
    // downloaded ones to: a ring of chunks, each reused once the work queued
    // on it has passed.  An admitted problem of 2300 nodes takes 10 us and a
    // downloaded one 21; three blocking copies from pageable memory and a
    // wait took 57, a device-side pack and a blocking copy 33.  8 MiB keep
    // the link busy: a chunk takes 40 us on it and 150 to fill.
    char* pin = nullptr;
    hipEvent_t pin_done[kPinChunks] = {};
    bool pin_busy[kPinChunks] = {};
    int pin_at = 0;
    size_t pin_used = 0;
    ItemArgs* d_items = nullptr;
    double* d_dt = nullptr;
    unsigned long long* d_dtmin = nullptr;
    double* d_time = nullptr;
    long long* d_steps = nullptr;
    long long* d_target = nullptr;
    unsigned* d_flags = nullptr;
    int* d_live = nullptr;
    BatchTile* d_tiles = nullptr;
    int* d_active = nullptr;
    int* d_scan = nullptr;
    size_t tile_cap = 0;
    // launch shape (tunable)
    int xlen = 0;               // nodes of a 1D tile, in strips of 63 (0: by cost)
    int ylen = 0;               // rows of a 2D tile (0: by cost)
    int blocks_per_cu = -1;     // persistent grid size (-1: a block per tile)
    int fused = 1;              // 1: one launch per stage for all variants
    // host side
    std::vector<Item> items;
    std::vector<sf_batch_item> desc;
    std::vector<char> used;
    std::map<long long, long long> free_ranges;  // offset -> length
    std::vector<int> pending_scan;               // admitted since the last step
    bool tables_dirty = true;
    int nactive = 0;
    int line[5] = {0, 0, 0, 0, 0}, plane[5] = {0, 0, 0, 0, 0};  // tile ranges per variant
    bool any2d = false;
    hipGraph_t graph = nullptr;
    hipGraphExec_t graph_exec = nullptr;
};

namespace {

BatchDev view(const sf_batch* b) {
    BatchDev B{};
    B.items = b->d_items;
    B.active = b->d_active;
    B.nactive = b->nactive;
    B.dt = b->d_dt;
    B.dtmin = b->d_dtmin;
    B.time = b->d_time;
    B.steps = b->d_steps;
    B.target = b->d_target;
    B.flags = b->d_flags;
    B.live = b->d_live;
    return B;
}

// Arguments of the three stages of a problem in slot `slot`: stage s reads
// buf[s] and writes buf[s + 1], the last one buf[0].  Uniform Cartesian
// metrics are formed as for a grid with unit spacing on the absent axes
// (SF_mesh.cpp:320-338, SF_canonicalFace.h:87-108).
ItemArgs item_args(const sf_batch* b, int slot, const sf_batch::Item& it,
                   const sf_batch_item* item) {
    SweepArgs W{};
    GridDev& G = W.G;
    const int n[3] = {it.n0, it.n1, 1};
    const int ghosts[3] = {3, it.gy, 0};
    const double d[3] = {item->d[0], it.n1 > 1 ? item->d[1] : 1.0, 1.0};
    G.jac = 1.0 / (d[0] * d[1] * d[2]);
    for (int a = 0; a < 3; ++a) {
        const int on = n[a] > 1;
        G.n[a] = n[a];
        G.g[a] = ghosts[a];
        G.m[a] = n[a] + 2 * ghosts[a];
        G.active[a] = on;
        G.zg_lo[a] = G.zg_hi[a] = on;
        G.solved_lo[a] = on;
        G.solved_hi[a] = n[a] - 1 - on;
        G.map_lo[a] = on ? -1 : std::numeric_limits<int>::min();
        G.map_hi[a] = on ? n[a] : std::numeric_limits<int>::max();
        G.d[a] = d[a];
        const double metric = 1.0 / d[a];
        const double c = metric / G.jac, f = 0.5 * (c + c);
        G.area[a] = std::sqrt(f * f + 0.0 * 0.0 + 0.0 * 0.0);
        G.metric[a] = on ? metric : 0.0;
    }
    G.xo = 3;
    G.P = b->capacity;
    G.stride[0] = 1;
    G.stride[1] = it.m0;
    G.stride[2] = (long long)it.m0 * G.m[1];
    for (int a = 0; a < 3; ++a) G.ustride[a] = (unsigned)G.stride[a];
    G.gamma = b->gamma;
    static const double base[3] = {0.0, 0.75, 1.0 / 3.0};
    static const double incr[3] = {1.0, 0.25, 2.0 / 3.0};
    W.A.q0 = b->buf[0] + it.off;
    W.A.dt = b->d_dt + slot;
    W.A.dtmin = b->d_dtmin + (size_t)slot * kItemDtWords;
    W.A.flags = b->d_flags + slot;
    W.A.cfl = item->cfl;
    W.A.time = SF_TIME_SSPRK3;
    ItemArgs args{};
    for (int s = 0; s < 3; ++s) {
        W.q = b->buf[s] + it.off;
        W.A.qout = b->buf[(s + 1) % 3] + it.off;
        W.A.base = base[s];
        W.A.incr = incr[s];
        W.A.stage = s;
        W.A.reduce_dt = s == 2;
        args.stage[s] = W;
    }
    return args;
}

void drop_graph(sf_batch* b) {
    if (b->graph_exec) (void)hipGraphExecDestroy(b->graph_exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    b->graph_exec = nullptr;
    b->graph = nullptr;
}

int pin_open(sf_batch* b) {
    if (b->pin) return 0;
    for (hipEvent_t& e : b->pin_done)
        if (!e) SF_BHIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    SF_BHIP(hipHostMalloc((void**)&b->pin, kPinChunks * kPinBytes, hipHostMallocDefault));
    return 0;
}

// Room for `bytes` (at most a chunk) in the pinned ring.  The work on it has
// to be queued on the compute stream before the next call.
int pin_reserve(sf_batch* b, size_t bytes, void** out) {
    if (int rc = pin_open(b)) return rc;
    if (b->pin_used + bytes > kPinBytes) {
        SF_BHIP(hipEventRecord(b->pin_done[b->pin_at], b->stream));
        b->pin_busy[b->pin_at] = true;
        b->pin_at = (b->pin_at + 1) % kPinChunks;
        if (b->pin_busy[b->pin_at]) SF_BHIP(hipEventSynchronize(b->pin_done[b->pin_at]));
        b->pin_busy[b->pin_at] = false;
        b->pin_used = 0;
    }
    *out = b->pin + b->pin_at * kPinBytes + b->pin_used;
    b->pin_used += (bytes + 255) & ~(size_t)255;
    return 0;
}

// The compute stream is idle: the whole ring is free.
void pin_reset(sf_batch* b) {
    for (bool& busy : b->pin_busy) busy = false;
    b->pin_used = 0;
}

// Queue a copy of host data that may be changed on return.
int upload(sf_batch* b, void* dst, const void* src, size_t bytes) {
    for (size_t o = 0; o < bytes; o += kPinBytes) {
        const size_t n = std::min(kPinBytes, bytes - o);
        void* p = nullptr;
        if (int rc = pin_reserve(b, n, &p)) return rc;
        std::memcpy(p, (const char*)src + o, n);
        SF_BHIP(hipMemcpyAsync((char*)dst + o, p, n, hipMemcpyHostToDevice, b->stream));
    }
    return 0;
}

// Strips of a 2D problem along x: 63 columns and a lane that evaluates the
// first face, or 64 with the first faces evaluated beforehand where that
// saves a strip.
struct Strips {
    int cols, count;
};

Strips strips(int n0) {
    const int nx = n0 - 2;
    const Strips s{kXBlock - 1, (nx + kXBlock - 2) / (kXBlock - 1)};
    const int whole = (nx + kXBlock - 1) / kXBlock;
    return whole < s.count ? Strips{kXBlock, whole} : s;
}

// Tile table and the active list after admissions / removals.  Tiles are
// grouped by (scheme, flux) variant and, within a variant, listed largest
// problem first, so the blocks start on the big problems and finish on the
// small ones.  Rows of a 2D tile and strips of a 1D one are the longest that
// march_cost finds worth while over all problems of the kind: few problems
// then spread over the whole device, many run long tiles.  A node's
// arithmetic does not depend on them.
int rebuild_tables(sf_batch* b) {
    std::vector<int> act;
    b->any2d = false;
    for (int s = 0; s < b->item_capacity; ++s)
        if (b->used[s]) act.push_back(s);
    std::vector<int> order = act;
    auto variant = [&](int s) { return 2 * b->items[s].scheme + b->items[s].flux; };
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
        if (variant(x) != variant(y)) return variant(x) < variant(y);
        return (long long)b->items[x].n0 * b->items[x].n1 >
               (long long)b->items[y].n0 * b->items[y].n1;
    });
    const auto line_strips = [&](int s) { return (b->items[s].n0 - 2 + kXBlock - 2) / (kXBlock - 1); };
    // the least cost over tile lengths 1 .. most
    const auto choose = [&](int most, double faces_per, double extra, auto tiles_of) {
        int best = 1;
        double least = 0.0;
        for (int r = 1; r <= most; ++r) {
            long long blocks = 0;
            for (int s : order) blocks += tiles_of(s, r);
            const double cost = march_cost(blocks, faces_per * r + extra, b->cus);
            if (r > 1 && cost >= least) continue;
            least = cost;
            best = r;
        }
        return best;
    };
    for (int s : order) b->any2d = b->any2d || b->items[s].n1 > 1;
    int rows = std::min(b->ylen, kYxRows), run = (b->xlen + 1) / kXBlock;
    if (b->any2d && rows == 0)
        rows = choose(kYxRows, 2.0, 1.0, [&](int s, int r) -> long long {
            const sf_batch::Item& it = b->items[s];
            return it.n1 > 1 ? (long long)strips(it.n0).count * ((it.n1 - 2 + r - 1) / r) : 0;
        });
    if (run == 0)
        run = choose(8, 1.0, 0.0, [&](int s, int r) -> long long {
            return b->items[s].n1 > 1 ? 0 : (line_strips(s) + r - 1) / r;
        });
    std::vector<BatchTile> tiles;
    const auto fill = [&](bool plane, int (&range)[5]) {
        int v = 0;
        range[0] = (int)tiles.size();
        for (int s : order) {
            const sf_batch::Item& it = b->items[s];
            if ((it.n1 > 1) != plane) continue;
            while (v < variant(s)) range[++v] = (int)tiles.size();
            if (plane) {
                const Strips st = strips(it.n0);
                const int helper = kXBlock - st.cols;
                for (int a0 = 1; a0 <= it.n1 - 2; a0 += rows)
                    for (int x = 0; x < st.count; ++x)
                        tiles.push_back({s, 1 + x * st.cols - helper, a0,
                                         (int)((unsigned)std::min(a0 + rows, it.n1 - 1) |
                                               ((unsigned)helper << 31))});
            } else {
                for (int x = 0; x < line_strips(s); x += run)
                    tiles.push_back({s, x * (kXBlock - 1), run, 0});
            }
        }
        while (v < 4) range[++v] = (int)tiles.size();
    };
    fill(true, b->plane);
    fill(false, b->line);
    if (tiles.size() > b->tile_cap) {
        if (b->d_tiles) SF_BHIP(hipFree(b->d_tiles));
        b->d_tiles = nullptr;
        b->tile_cap = 0;
        const size_t want = std::max<size_t>(tiles.size(), 1024);
        SF_BHIP(hipMalloc(&b->d_tiles, want * sizeof(BatchTile)));
        b->tile_cap = want;
    }
    if (int rc = upload(b, b->d_tiles, tiles.data(), tiles.size() * sizeof(BatchTile))) return rc;
    if (int rc = upload(b, b->d_active, act.data(), act.size() * sizeof(int))) return rc;
    b->nactive = (int)act.size();
    b->tables_dirty = false;
    drop_graph(b);
    return 0;
}

// Relative cost of a tile of each variant (TENO5 evaluates its three
// candidate weights with a sixth power; HLLC adds a star state).
constexpr double kVariantCost[4] = {1.0, 1.08, 1.52, 1.62};

// Block ranges of a fused launch of `total` blocks over the variant tile
// ranges r[5]: proportional to the tiles' cost, at least one block for a
// non-empty variant, never more blocks than tiles.
Split split_blocks(const int r[5], unsigned total) {
    Split sp{};
    const unsigned tiles = (unsigned)(r[4] - r[0]);
    double w[4], sum = 0.0;
    for (int v = 0; v < 4; ++v) {
        w[v] = (r[v + 1] - r[v]) * kVariantCost[v];
        sum += w[v];
    }
    sp.tile[0] = r[0];
    sp.block[0] = 0;
    for (int v = 0; v < 4; ++v) {
        const int n = r[v + 1] - r[v];
        int nb = 0;
        if (total >= tiles) nb = n;
        else if (n > 0) nb = std::min(n, std::max(1, (int)std::lround(total * w[v] / sum)));
        sp.tile[v + 1] = r[v + 1];
        sp.block[v + 1] = sp.block[v] + nb;
    }
    return sp;
}

// Blocks of `kernel` (block size `threads`) a compute unit holds at once,
// from the runtime's occupancy calculator (cached per kernel).
template <class Kernel>
int resident_per_cu(Kernel kernel, int threads) {
    static std::map<const void*, int> cache;
    static std::mutex mu;
    std::lock_guard<std::mutex> lock(mu);
    const void* key = reinterpret_cast<const void*>(kernel);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, threads, 0) != hipSuccess || n < 1)
        n = 4;
    cache[key] = n;
    return n;
}

// Grid of a stage over `tiles` tiles: a block per tile, or persistent
// blocks, blocks_per_cu per compute unit, or with blocks_per_cu = 0 as many
// as the device holds at once.  A block per tile is the default: the
// dispatcher hands the next tile to whichever SIMD is free.
template <class Kernel>
unsigned stage_blocks(const sf_batch* b, int tiles, Kernel kernel) {
    if (b->blocks_per_cu < 0) return (unsigned)tiles;
    const int want = b->blocks_per_cu > 0 ? b->blocks_per_cu : resident_per_cu(kernel, kXBlock);
    return (unsigned)std::max(1, std::min(tiles, b->cus * want));
}

template <bool PLANE, int SCHEME, int FLUX>
void launch_variant(sf_batch* b, const BatchStage& B, const int r[5]) {
    constexpr int v = 2 * SCHEME + FLUX;
    if (r[v + 1] == r[v]) return;
    k_batch_stage<PLANE, SCHEME, FLUX>
        <<<stage_blocks(b, r[v + 1] - r[v], k_batch_stage<PLANE, SCHEME, FLUX>), kXBlock, 0,
           b->stream>>>(B, r[v], r[v + 1]);
}

// Stage of the 2D (PLANE) or the 1D problems.  With one variant present the
// kernel of its own is the fused launch, too.
template <bool PLANE>
void launch_stage(sf_batch* b, const BatchStage& B, const int r[5]) {
    int present = 0;
    for (int v = 0; v < 4; ++v) present += r[v + 1] > r[v];
    if (b->fused && present > 1) {
        const Split sp =
            split_blocks(r, stage_blocks(b, r[4] - r[0], k_batch_stage_mixed<PLANE>));
        k_batch_stage_mixed<PLANE><<<(unsigned)sp.block[4], kXBlock, 0, b->stream>>>(B, sp);
        return;
    }
    launch_variant<PLANE, 0, 0>(b, B, r);
    launch_variant<PLANE, 0, 1>(b, B, r);
    launch_variant<PLANE, 1, 0>(b, B, r);
    launch_variant<PLANE, 1, 1>(b, B, r);
}

void launch_clock(sf_batch* b, int next) {
    k_batch_clock<<<(unsigned)((b->nactive + 63) / 64), 64, 0, b->stream>>>(view(b), next);
}

// One SSPRK3 step of every live problem (the captured sequence); its commit
// is the next clock launch.
void enqueue_step(sf_batch* b) {
    launch_clock(b, 1);
    for (int s = 0; s < 3; ++s) {
        const BatchStage B{b->d_items, b->d_live, b->d_tiles, s};
        launch_stage<true>(b, B, b->plane);
        launch_stage<false>(b, B, b->line);
    }
}

int check_item(const sf_batch_item* it) {
    if (!it) return bfail(SF_E_ARG, "null batch item");
    if (it->n[0] < 4) return bfail(SF_E_ARG, "a batch problem needs at least 4 nodes along x");
    if (it->n[1] != 1 && it->n[1] < 4)
        return bfail(SF_E_ARG, "a 2D batch problem needs at least 4 nodes along y");
    if (!(it->d[0] > 0.0) || (it->n[1] > 1 && !(it->d[1] > 0.0)))
        return bfail(SF_E_ARG, "node spacing must be positive");
    if (it->scheme != SF_SCHEME_WENO5 && it->scheme != SF_SCHEME_TENO5)
        return bfail(SF_E_ARG, "the batch serves the WENO5 and TENO5 reconstructions "
                               "(WENO3 and WENO7 run on the grid path)");
    if (it->flux != SF_FLUX_RUSANOV && it->flux != SF_FLUX_HLLC)
        return bfail(SF_E_ARG, "the batch serves the Rusanov and HLLC fluxes (Steger-Warming, "
                               "Lax-Friedrichs and Roe run on the grid path)");
    if (!(it->cfl > 0.0) || !std::isfinite(it->cfl)) return bfail(SF_E_ARG, "invalid CFL number");
    return 0;
}

bool valid_slot(const sf_batch* b, int slot) {
    return b && slot >= 0 && slot < b->item_capacity && b->used[slot];
}

// Boundary nodes and CFL scan of the problems admitted since the last step.
int prepare_pending(sf_batch* b) {
    if (b->pending_scan.empty()) return 0;
    const int n = (int)b->pending_scan.size();
    if (int rc = upload(b, b->d_scan, b->pending_scan.data(), sizeof(int) * (size_t)n)) return rc;
    const BatchDev B = view(b);
    k_batch_reset<<<(n + 255) / 256, 256, 0, b->stream>>>(B, b->d_scan, n);
    const dim3 grid((unsigned)n, 16);
    k_batch_prepare<<<grid, 256, 0, b->stream>>>(B, b->d_scan);
    SF_BHIP(hipGetLastError());
    b->pending_scan.clear();
    return 0;
}

// Steps of a captured graph.  A replay costs 6 us between graphs, which a
// step of its own four launches does not: 300 nodes took 25 us per step in
// graphs of one step and take 18.7 in graphs of eight, 18.6 launched directly;
// 131^2 41, 34 and 34.
constexpr int kGraphSteps = 8;

// Queue nsteps steps (graph replays and, for the rest, direct launches); no
// wait.  Left to choose (2), direct launches: they are as fast on the device
// and need no capture.
int advance(sf_batch* b, int nsteps, int use_graph) {
    int s = 0;
    if (use_graph == 1 && nsteps >= kGraphSteps) {
        if (!b->graph_exec) {
            SF_BHIP(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
            for (int k = 0; k < kGraphSteps; ++k) enqueue_step(b);
            hipGraph_t g = nullptr;
            SF_BHIP(hipStreamEndCapture(b->stream, &g));
            b->graph = g;
            SF_BHIP(hipGraphInstantiate(&b->graph_exec, g, nullptr, nullptr, 0));
        }
        for (; s + kGraphSteps <= nsteps; s += kGraphSteps)
            SF_BHIP(hipGraphLaunch(b->graph_exec, b->stream));
    }
    for (; s < nsteps; ++s) enqueue_step(b);
    launch_clock(b, 0);
    SF_BHIP(hipGetLastError());
    return 0;
}

// Per-problem fault flags of the admitted problems (0 for free slots);
// returns the number of faulted problems.
int read_faults(sf_batch* b, unsigned* flags, int* faulted) {
    SF_BHIP(hipMemcpy(flags, b->d_flags, sizeof(unsigned) * b->item_capacity,
                      hipMemcpyDeviceToHost));
    int n = 0;
    for (int s = 0; s < b->item_capacity; ++s) {
        if (!b->used[s]) flags[s] = 0;
        n += flags[s] != 0;
    }
    *faulted = n;
    return 0;
}

}  // namespace

extern "C" {

int sf_batch_item_nodes(const sf_batch_item* item, size_t* nodes) {
    if (int rc = check_item(item)) return rc;
    if (nodes) *nodes = (size_t)padded_nodes(*item);
    return 0;
}

int sf_batch_create(int device, double gamma, size_t node_capacity, int item_capacity,
                    sf_batch** out) {
    if (!out) return bfail(SF_E_ARG, "sf_batch_create: null output");
    *out = nullptr;
    if (!(gamma > 1.0)) return bfail(SF_E_ARG, "gamma must exceed 1");
    if (node_capacity < 64 || item_capacity < 1)
        return bfail(SF_E_ARG, "sf_batch_create: capacities must be positive");
    int ndev = 0;
    SF_BHIP(hipGetDeviceCount(&ndev));
    if (device < 0 || device >= ndev) return bfail(SF_E_ARG, "device ordinal out of range");
    SF_BHIP(hipSetDevice(device));
    sf_batch* b = new (std::nothrow) sf_batch;
    if (!b) return bfail(SF_E_MEMORY, "host allocation failed");
    b->device = device;
    b->gamma = gamma;
    b->capacity = (long long)node_capacity;
    b->item_capacity = item_capacity;
    if (hipDeviceGetAttribute(&b->cus, hipDeviceAttributeMultiprocessorCount, device) !=
            hipSuccess || b->cus <= 0)
        b->cus = 256;   // MI355X's CU count; only the launch shapes depend on it
    const size_t state = sizeof(double) * 5 * node_capacity;
    bool ok = true;
    for (int i = 0; i < 3 && ok; ++i) ok = hipMalloc(&b->buf[i], state) == hipSuccess;
    ok = ok && hipMalloc(&b->d_items, sizeof(ItemArgs) * item_capacity) == hipSuccess;
    ok = ok && hipMalloc(&b->d_dt, sizeof(double) * item_capacity) == hipSuccess;
    ok = ok && hipMalloc(&b->d_dtmin, sizeof(unsigned long long) * kItemDtWords * item_capacity) == hipSuccess;
    ok = ok && hipMalloc(&b->d_time, sizeof(double) * item_capacity) == hipSuccess;
    ok = ok && hipMalloc(&b->d_steps, sizeof(long long) * item_capacity) == hipSuccess;
    ok = ok && hipMalloc(&b->d_target, sizeof(long long) * item_capacity) == hipSuccess;
    ok = ok && hipMalloc(&b->d_flags, sizeof(unsigned) * item_capacity) == hipSuccess;
    ok = ok && hipMalloc(&b->d_live, sizeof(int) * item_capacity) == hipSuccess;
    ok = ok && hipMalloc(&b->d_active, sizeof(int) * item_capacity) == hipSuccess;
    ok = ok && hipMalloc(&b->d_scan, sizeof(int) * item_capacity) == hipSuccess;
    ok = ok && hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) == hipSuccess;
    ok = ok && hipStreamCreateWithFlags(&b->copy_stream, hipStreamNonBlocking) == hipSuccess;
    ok = ok && hipEventCreateWithFlags(&b->copy_after, hipEventDisableTiming) == hipSuccess;
    // cleared on the stream that uses them: the first admission is not waited
    // for, and the compute stream does not wait for the null stream
    const auto clear = [&](void* p, size_t bytes) {
        return hipMemsetAsync(p, 0, bytes, b->stream) == hipSuccess;
    };
    ok = ok && clear(b->d_flags, sizeof(unsigned) * item_capacity);
    ok = ok && clear(b->d_live, sizeof(int) * item_capacity);
    ok = ok && clear(b->d_steps, sizeof(long long) * item_capacity);
    ok = ok && clear(b->d_target, sizeof(long long) * item_capacity);
    // the arena starts zeroed, so padding that is never written stays finite
    for (int i = 0; i < 3 && ok; ++i) ok = clear(b->buf[i], state);
    if (!ok) {
        sf_batch_destroy(b);
        return bfail(SF_E_MEMORY, "sf_batch_create: device allocation of " +
                                      std::to_string(3 * state) + " bytes failed");
    }
    b->items.resize(item_capacity);
    b->desc.resize(item_capacity);
    b->used.assign(item_capacity, 0);
    b->free_ranges[0] = (long long)node_capacity;
    *out = b;
    return 0;
}

int sf_batch_destroy(sf_batch* b) {
    if (!b) return 0;
    (void)hipSetDevice(b->device);
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    if (b->copy_stream) (void)hipStreamSynchronize(b->copy_stream);
    drop_graph(b);
    for (double* p : b->buf)
        if (p) (void)hipFree(p);
    if (b->pin) (void)hipHostFree(b->pin);
    for (hipEvent_t e : b->pin_done)
        if (e) (void)hipEventDestroy(e);
    void* ptrs[] = {b->d_items, b->d_dt,   b->d_dtmin, b->d_time,   b->d_steps, b->d_target,
                    b->d_flags, b->d_live, b->d_tiles, b->d_active, b->d_scan};
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    if (b->stream) (void)hipStreamDestroy(b->stream);
    if (b->copy_stream) (void)hipStreamDestroy(b->copy_stream);
    if (b->copy_after) (void)hipEventDestroy(b->copy_after);
    delete b;
    return 0;
}


int sf_batch_add(sf_batch* b, const sf_batch_item* item, const double* soa, long long max_steps,
                 int* slot) {
    if (!b || !soa || !slot) return bfail(SF_E_ARG, "sf_batch_add: null argument");
    if (int rc = check_item(item)) return rc;
    if (max_steps < 0) return bfail(SF_E_ARG, "sf_batch_add: negative step limit");
    SF_BHIP(hipSetDevice(b->device));
    const long long need = padded_nodes(*item);
    auto fit = b->free_ranges.end();
    for (auto it = b->free_ranges.begin(); it != b->free_ranges.end(); ++it)
        if (it->second >= need) {
            fit = it;
            break;
        }
    int s = -1;
    for (int k = 0; k < b->item_capacity; ++k)
        if (!b->used[k]) {
            s = k;
            break;
        }
    if (s < 0) return bfail(SF_E_MEMORY, "sf_batch_add: every problem slot is taken");
    if (fit == b->free_ranges.end())
        return bfail(SF_E_MEMORY, "sf_batch_add: no room in the arena for the problem (" +
                                      std::to_string(need) + " padded nodes)");
    const long long N = (long long)item->n[0] * std::max(1, item->n[1]);
    const long long off = fit->first, len = fit->second;
    sf_batch::Item it;
    it.off = off;
    it.n0 = item->n[0];
    it.n1 = std::max(1, item->n[1]);
    it.m0 = it.n0 + 6;
    it.gy = it.n1 > 1 ? 3 : 0;
    it.scheme = item->scheme;
    it.flux = item->flux;
    const ItemArgs args = item_args(b, s, it, item);
    const long long target = max_steps > 0 ? max_steps : LLONG_MAX;
    for (long long u0 = 0; u0 < N; u0 += kPinNodes) {
        const long long cnt = std::min(kPinNodes, N - u0);
        void* p = nullptr;
        if (int rc = pin_reserve(b, sizeof(double) * 5 * (size_t)cnt, &p)) return rc;
        for (int v = 0; v < 5; ++v)
            std::memcpy((double*)p + v * cnt, soa + v * N + u0, sizeof(double) * (size_t)cnt);
        k_batch_admit<<<(unsigned)((cnt + 255) / 256), 256, 0, b->stream>>>(
            args, b->d_items + s, b->d_target + s, target, (const double*)p, (unsigned)u0,
            (unsigned)cnt);
        SF_BHIP(hipGetLastError());
    }
    b->items[s] = it;
    b->free_ranges.erase(fit);
    if (len > need) b->free_ranges[off + need] = len - need;
    b->desc[s] = *item;
    b->used[s] = 1;
    b->pending_scan.push_back(s);
    b->tables_dirty = true;
    *slot = s;
    return 0;
}

int sf_batch_remove(sf_batch* b, int slot) {
    if (!valid_slot(b, slot)) return bfail(SF_E_ARG, "sf_batch_remove: invalid slot");
    SF_BHIP(hipSetDevice(b->device));
    SF_BHIP(hipStreamSynchronize(b->stream));
    b->used[slot] = 0;
    b->pending_scan.erase(std::remove(b->pending_scan.begin(), b->pending_scan.end(), slot),
                          b->pending_scan.end());
    long long off = b->items[slot].off, len = padded_nodes(b->desc[slot]);
    auto next = b->free_ranges.lower_bound(off);
    if (next != b->free_ranges.end() && next->first == off + len) {
        len += next->second;
        b->free_ranges.erase(next);
    }
    auto prev = b->free_ranges.lower_bound(off);
    if (prev != b->free_ranges.begin()) {
        --prev;
        if (prev->first + prev->second == off) {
            off = prev->first;
            len += prev->second;
            b->free_ranges.erase(prev);
        }
    }
    b->free_ranges[off] = len;
    b->tables_dirty = true;
    return 0;
}

int sf_batch_download(sf_batch* b, int slot, double* soa) {
    if (!soa || !valid_slot(b, slot)) return bfail(SF_E_ARG, "sf_batch_download: invalid slot");
    SF_BHIP(hipSetDevice(b->device));
    const sf_batch::Item& it = b->items[slot];
    const long long N = (long long)it.n0 * it.n1;
    if (int rc = pin_open(b)) return rc;
    // a chunk of the ring per piece; the pieces after it are written while
    // one is copied out
    const long long pieces = (N + kPinNodes - 1) / kPinNodes;
    const auto count = [&](long long p) { return std::min(kPinNodes, N - p * kPinNodes); };
    const auto chunk = [&](long long p) {
        return (double*)(b->pin + (size_t)(p % kPinChunks) * kPinBytes);
    };
    for (long long p = 0; p < pieces + kPinChunks; ++p) {
        const long long out = p - kPinChunks;
        if (out >= 0 && out < pieces) {
            if (pieces == 1) SF_BHIP(hipStreamSynchronize(b->stream));
            else SF_BHIP(hipEventSynchronize(b->pin_done[out % kPinChunks]));
            for (int v = 0; v < 5; ++v)
                std::memcpy(soa + v * N + out * kPinNodes, chunk(out) + v * count(out),
                            sizeof(double) * (size_t)count(out));
        }
        if (p < pieces) {
            k_batch_pack<<<(unsigned)((count(p) + 255) / 256), 256, 0, b->stream>>>(
                b->d_items + slot, chunk(p), (unsigned)(p * kPinNodes), (unsigned)count(p),
                nullptr);
            SF_BHIP(hipGetLastError());
            if (pieces > 1) SF_BHIP(hipEventRecord(b->pin_done[p % kPinChunks], b->stream));
        }
    }
    pin_reset(b);
    return 0;
}

int sf_batch_step(sf_batch* b, int nsteps, int use_graph) {
    if (!b || nsteps < 0 || use_graph < 0 || use_graph > 2)
        return bfail(SF_E_ARG, "sf_batch_step: invalid argument");
    SF_BHIP(hipSetDevice(b->device));
    if (b->tables_dirty)
        if (int rc = rebuild_tables(b)) return rc;
    if (int rc = prepare_pending(b)) return rc;
    if (b->nactive == 0 || nsteps == 0) return 0;
    if (int rc = advance(b, nsteps, use_graph)) return rc;
    SF_BHIP(hipStreamSynchronize(b->stream));
    pin_reset(b);
    std::vector<unsigned> flags((size_t)b->item_capacity);
    int faulted = 0;
    if (int rc = read_faults(b, flags.data(), &faulted)) return rc;
    if (faulted) {
        int first = 0;
        while (!flags[first]) ++first;
        char msg[200];
        std::snprintf(msg, sizeof msg,
                      "sf_batch_step: %d problem(s) raised numerical fault flags (slot %d: 0x%x); "
                      "they are frozen, the others advanced",
                      faulted, first, flags[first]);
        return bfail(SF_E_NUMERIC, msg);
    }
    return 0;
}

int sf_batch_faults(sf_batch* b, uint32_t* flags) {
    if (!b || !flags) return bfail(SF_E_ARG, "sf_batch_faults: null argument");
    SF_BHIP(hipSetDevice(b->device));
    SF_BHIP(hipStreamSynchronize(b->stream));
    int faulted = 0;
    return read_faults(b, flags, &faulted);
}

int sf_batch_clock(sf_batch* b, int slot, double* time, long long* steps) {
    if (!valid_slot(b, slot)) return bfail(SF_E_ARG, "sf_batch_clock: invalid slot");
    SF_BHIP(hipSetDevice(b->device));
    SF_BHIP(hipStreamSynchronize(b->stream));
    if (time) SF_BHIP(hipMemcpy(time, b->d_time + slot, sizeof(double), hipMemcpyDeviceToHost));
    if (steps)
        SF_BHIP(hipMemcpy(steps, b->d_steps + slot, sizeof(long long), hipMemcpyDeviceToHost));
    return 0;
}

int sf_batch_steps(sf_batch* b, long long* steps) {
    if (!b || !steps) return bfail(SF_E_ARG, "sf_batch_steps: null argument");
    SF_BHIP(hipSetDevice(b->device));
    SF_BHIP(hipStreamSynchronize(b->stream));
    SF_BHIP(hipMemcpy(steps, b->d_steps, sizeof(long long) * b->item_capacity,
                      hipMemcpyDeviceToHost));
    for (int s = 0; s < b->item_capacity; ++s)
        if (!b->used[s]) steps[s] = -1;
    return 0;
}

int sf_batch_memory(const sf_batch* b, size_t* used_nodes, size_t* free_nodes, int* items) {
    if (!b) return bfail(SF_E_ARG, "sf_batch_memory: null batch");
    long long fr = 0;
    for (const auto& kv : b->free_ranges) fr += kv.second;
    if (used_nodes) *used_nodes = (size_t)(b->capacity - fr);
    if (free_nodes) *free_nodes = (size_t)fr;
    if (items) *items = (int)std::count(b->used.begin(), b->used.end(), 1);
    return 0;
}

int sf_batch_set_tiles(sf_batch* b, int xlen, int ylen) {
    if (!b) return bfail(SF_E_ARG, "sf_batch_set_tiles: null batch");
    if (xlen != 0 && xlen != 63 && xlen != 127 && xlen != 255)
        return bfail(SF_E_ARG, "sf_batch_set_tiles: x tile must be 63, 127 or 255 nodes, or 0");
    if (ylen != 0 && (ylen < 4 || ylen > 4096))
        return bfail(SF_E_ARG, "sf_batch_set_tiles: y tile out of range");
    b->xlen = xlen;
    b->ylen = ylen;
    b->tables_dirty = true;
    return 0;
}

}  // extern "C"

// ---- autotuner ----------------------------------------------------------------
// Times launch shapes (schedule x x-tile x y-tile x persistent grid size) on
// the batch's own problems: each trial takes the same steps from the same
// saved state, which is restored afterwards, so tuning leaves the problems
// exactly as it found them.  The shape that the batch has, the automatic one
// unless it was set, is timed first and kept unless another is faster; what
// the batch holds no problems for keeps its setting.  Trials launch directly:
// a captured graph would be charged with its capture.
namespace {

struct Snapshot {
    double* q = nullptr;
    long long extent = 0;
    std::vector<double> dt, time;
    std::vector<unsigned long long> dtmin;
    std::vector<long long> steps;
    std::vector<unsigned> flags;
};

int snapshot_save(sf_batch* b, Snapshot& sn) {
    sn.extent = 0;
    for (int s = 0; s < b->item_capacity; ++s)
        if (b->used[s])
            sn.extent = std::max(sn.extent, b->items[s].off + padded_nodes(b->desc[s]));
    SF_BHIP(hipMalloc(&sn.q, sizeof(double) * 5 * (size_t)std::max(1LL, sn.extent)));
    for (int v = 0; v < 5; ++v)
        SF_BHIP(hipMemcpyAsync(sn.q + v * sn.extent, b->buf[0] + v * b->capacity,
                               sizeof(double) * sn.extent, hipMemcpyDeviceToDevice, b->stream));
    const size_t n = (size_t)b->item_capacity;
    sn.dt.resize(n);
    sn.time.resize(n);
    sn.dtmin.resize(n * kItemDtWords);
    sn.steps.resize(n);
    sn.flags.resize(n);
    SF_BHIP(hipStreamSynchronize(b->stream));
    SF_BHIP(hipMemcpy(sn.dt.data(), b->d_dt, sizeof(double) * n, hipMemcpyDeviceToHost));
    SF_BHIP(hipMemcpy(sn.time.data(), b->d_time, sizeof(double) * n, hipMemcpyDeviceToHost));
    SF_BHIP(hipMemcpy(sn.dtmin.data(), b->d_dtmin, 8 * n * kItemDtWords, hipMemcpyDeviceToHost));
    SF_BHIP(hipMemcpy(sn.steps.data(), b->d_steps, 8 * n, hipMemcpyDeviceToHost));
    SF_BHIP(hipMemcpy(sn.flags.data(), b->d_flags, 4 * n, hipMemcpyDeviceToHost));
    return 0;
}

int snapshot_restore(sf_batch* b, const Snapshot& sn) {
    for (int v = 0; v < 5; ++v)
        SF_BHIP(hipMemcpyAsync(b->buf[0] + v * b->capacity, sn.q + v * sn.extent,
                               sizeof(double) * sn.extent, hipMemcpyDeviceToDevice, b->stream));
    SF_BHIP(hipStreamSynchronize(b->stream));
    const size_t n = (size_t)b->item_capacity;
    SF_BHIP(hipMemcpy(b->d_dt, sn.dt.data(), sizeof(double) * n, hipMemcpyHostToDevice));
    SF_BHIP(hipMemcpy(b->d_time, sn.time.data(), sizeof(double) * n, hipMemcpyHostToDevice));
    SF_BHIP(hipMemcpy(b->d_dtmin, sn.dtmin.data(), 8 * n * kItemDtWords, hipMemcpyHostToDevice));
    SF_BHIP(hipMemcpy(b->d_steps, sn.steps.data(), 8 * n, hipMemcpyHostToDevice));
    SF_BHIP(hipMemcpy(b->d_flags, sn.flags.data(), 4 * n, hipMemcpyHostToDevice));
    return 0;
}

// Mean time of one step of the current shape over `steps` steps (after an
// untimed one).
int time_shape(sf_batch* b, int steps, double* ms) {
    if (b->tables_dirty)
        if (int rc = rebuild_tables(b)) return rc;
    if (int rc = advance(b, 1, 0)) return rc;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    SF_BHIP(hipEventCreate(&e0));
    SF_BHIP(hipEventCreate(&e1));
    int rc = 0;
    if (hipEventRecord(e0, b->stream) != hipSuccess) rc = bfail(SF_E_HIP, "event record failed");
    if (!rc) rc = advance(b, steps, 0);
    if (!rc && hipEventRecord(e1, b->stream) != hipSuccess)
        rc = bfail(SF_E_HIP, "event record failed");
    if (!rc && hipEventSynchronize(e1) != hipSuccess) rc = bfail(SF_E_HIP, "event wait failed");
    float t = 0.0f;
    if (!rc && hipEventElapsedTime(&t, e0, e1) != hipSuccess)
        rc = bfail(SF_E_HIP, "event timing failed");
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    *ms = (double)t / steps;
    return rc;
}

}  // namespace

extern "C" int sf_batch_autotune(sf_batch* b, int trial_steps, sf_batch_tuning* out) {
    if (!b || !out || trial_steps < 1) return bfail(SF_E_ARG, "sf_batch_autotune: invalid argument");
    SF_BHIP(hipSetDevice(b->device));
    if (b->tables_dirty)
        if (int rc = rebuild_tables(b)) return rc;
    if (int rc = prepare_pending(b)) return rc;
    if (b->nactive == 0) return bfail(SF_E_STATE, "sf_batch_autotune: the batch is empty");
    Snapshot sn;
    int rc = snapshot_save(b, sn);
    using Shape = sf_batch_tuning;
    const auto set = [&](const Shape& sh) {
        b->xlen = sh.xlen;
        b->ylen = sh.ylen;
        b->blocks_per_cu = sh.blocks_per_cu;
        b->fused = sh.fused;
        b->tables_dirty = true;
    };
    const auto timed = [&](Shape& sh) {
        set(sh);
        if (int e = time_shape(b, trial_steps, &sh.ms_per_step)) return e;
        return snapshot_restore(b, sn);
    };
    const Shape own{b->xlen, b->ylen, b->blocks_per_cu, b->fused, 0.0, 0};
    Shape best = own;
    if (!rc) rc = timed(best);
    bool any1d = false;
    for (int s = 0; s < b->item_capacity; ++s) any1d = any1d || (b->used[s] && b->items[s].n1 == 1);
    int tried = 0;
    const std::vector<int> xlens = any1d ? std::vector<int>{63, 127, 255} : std::vector<int>{own.xlen};
    const std::vector<int> ylens = b->any2d ? std::vector<int>{8, 16, 32} : std::vector<int>{own.ylen};
    for (int fused = 0; fused < 2 && !rc; ++fused)
        for (int xl : xlens)
            for (int yl : ylens)
                for (int oc : {0, 2, 4, 8, 16}) {   // 0: as many as stay resident
                    if (rc) break;
                    Shape sh{xl, yl, oc, fused, 0.0, 0};
                    rc = timed(sh);
                    if (rc) break;
                    ++tried;
                    if (sh.ms_per_step < best.ms_per_step) best = sh;
                }
    if (sn.q) (void)hipFree(sn.q);
    set(rc ? own : best);
    if (rc) return rc;
    best.candidates = tried;
    *out = best;
    return 0;
}

extern "C" int sf_batch_set_schedule(sf_batch* b, int fused) {
    if (!b) return bfail(SF_E_ARG, "sf_batch_set_schedule: null batch");
    b->fused = fused ? 1 : 0;
    drop_graph(b);
    return 0;
}

extern "C" int sf_batch_set_occupancy(sf_batch* b, int blocks_per_cu) {
    if (!b) return bfail(SF_E_ARG, "sf_batch_set_occupancy: null batch");
    if (blocks_per_cu < -1 || blocks_per_cu > 64)
        return bfail(SF_E_ARG,
                     "sf_batch_set_occupancy: 1..64 workgroups per compute unit, 0 for as "
                     "many as stay resident, or -1 for one per tile");
    b->blocks_per_cu = blocks_per_cu;
    drop_graph(b);
    return 0;
}

namespace sfamd {

long long batch_copy_doubles(const sf_batch* b, int slot) {
    const sf_batch::Item& it = b->items[(size_t)slot];
    return 5LL * it.n0 * it.n1 + 1;
}

int batch_copy_out_async(sf_batch* b, int slot, double* dst, hipEvent_t done) {
    if (!valid_slot(b, slot)) return bfail(SF_E_ARG, "batch copy-out: invalid slot");
    SF_BHIP(hipSetDevice(b->device));
    const sf_batch::Item& it = b->items[(size_t)slot];
    const unsigned N = (unsigned)it.n0 * (unsigned)it.n1;
    SF_BHIP(hipEventRecord(b->copy_after, b->stream));
    SF_BHIP(hipStreamWaitEvent(b->copy_stream, b->copy_after, 0));
    k_batch_pack<<<(N + 255) / 256, 256, 0, b->copy_stream>>>(b->d_items + slot, dst, 0, N,
                                                              b->d_time + slot);
    SF_BHIP(hipGetLastError());
    SF_BHIP(hipEventRecord(done, b->copy_stream));
    return 0;
}

void batch_unpack(const sf_batch* b, int slot, const double* src, double* soa, double* time) {
    const sf_batch::Item& it = b->items[(size_t)slot];
    const size_t N = (size_t)it.n0 * (size_t)it.n1;
    std::memcpy(soa, src, sizeof(double) * 5 * N);
    *time = src[5 * N];
}

}  // namespace sfamd
