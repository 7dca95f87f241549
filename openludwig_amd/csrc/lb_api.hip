// lb_api.hip -- C ABI of libludwig_hip.so (declared in include/ludwig_hip.h).
//
// Host side of the time step: device state per level, the 2:1 multilevel
// recursion of execute_timestep_batch! / recursive_step!
// (src/solver/solver_control.jl:6-219), and the layout conversions between
// the reference's column-major arrays and the device's block-major SoA.
//
// Differences in data flow from the reference, each exact:
//   * f_old / vel_old / g_old are not copies: a level with children keeps its
//     step's input buffers (f_in, vel_in, g_in) untouched until its next step,
//     which comes after both child substeps, so the children read them in
//     place (copy_to_old!, src/geometry/blocks.jl:241-252).  rho and T, single
//     buffers in the reference, are ping-ponged by step parity so the previous
//     step's values survive as rho_old / T_old.
//   * f_post_collision is not allocated: Bouzidi gathers its inputs from the
//     uncorrected f_out before it stores the corrected slots.
//   * No device synchronisation between launches; everything is ordered on
//     the context's stream.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <condition_variable>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <unordered_map>
#include <vector>

#include "ludwig_hip.h"
#include "lb_kernels.h"
#include "lb_sync.h"

namespace {

constexpr int NC = 512;
constexpr int Q = 27;

struct Kern {
    hipError_t (*collide)(const lbk::LevelArgs*, const lbk::CaseState*, const lbk::Work*, int32_t, int64_t, int, int,
                          int, int, hipStream_t);
    hipError_t (*thermal)(const lbk::LevelArgs*, const lbk::CaseState*, const lbk::Work*, int32_t, int64_t, int, int,
                          int, hipStream_t);
    hipError_t (*ghost_fill)(const lbk::LevelArgs*, const lbk::CaseState*, const lbk::Work*, int32_t, int64_t, int,
                             hipStream_t);
    hipError_t (*bouzidi)(const lbk::LevelArgs*, const lbk::CaseState*, const lbk::Work*, int32_t, int64_t, int,
                          hipStream_t);
    hipError_t (*set_state)(lbk::CaseState*, const lbk::CaseState&, hipStream_t);
    hipError_t (*advance)(lbk::CaseState*, int32_t, hipStream_t);
    hipError_t (*init_level)(void*, void*, float*, float*, float*, float*, int32_t, int, hipStream_t);
    hipError_t (*init_thermal)(void*, void*, float*, float*, int32_t, float, int, hipStream_t);
    hipError_t (*forces)(const lbk::ForceArgs&, int, double*, hipStream_t);
    hipError_t (*stats)(const void*, const float*, const float*, const uint8_t*, int32_t, int, double*, int,
                        hipStream_t);
    hipError_t (*export_rows)(const void*, const int32_t*, int32_t, int32_t, int, int64_t, int32_t, float*, hipStream_t);
    hipError_t (*finite_count)(const lbk::FiniteEntry*, int32_t, int64_t, int32_t*, hipStream_t);
    hipError_t (*engine_forces)(const lbk::EngineForce*, const lbk::CaseState*, const lbk::Work*, int32_t,
                                const int32_t*, int32_t, int64_t, hipStream_t);
};

#define LBK_TABLE(NS)                                                                                     \
    {NS::collide, NS::thermal, NS::ghost_fill, NS::bouzidi, NS::set_state, NS::advance, NS::init_level,  \
     NS::init_thermal, NS::forces, NS::stats, NS::export_rows, NS::finite_count, NS::engine_forces}
const Kern kStrict = LBK_TABLE(lbk_strict);
const Kern kFast = LBK_TABLE(lbk_fast);

struct Level {
    bool uploaded = false;
    int id = 0;
    int32_t nb = 0;
    double dx = 0;
    float tau = 0, tau_g = 0;
    void* f[2] = {nullptr, nullptr};  // 4 or 2 bytes per population (lb_config.storage)
    float* rho[2] = {nullptr, nullptr};
    float* vel[2] = {nullptr, nullptr};
    void* g[2] = {nullptr, nullptr};  // thermal populations, same storage as f
    float* T[2] = {nullptr, nullptr};
    uint8_t* obst = nullptr;
    float* sponge = nullptr;
    float* wall_dist = nullptr;
    std::vector<int32_t> wflags;  // per block: WORK_* of its work entry
    int32_t* nbr = nullptr;
    int32_t* borg = nullptr;
    int32_t* inv = nullptr;  // caller's block -> device block
    int32_t* grid = nullptr;
    // ghost blocks (coarse-to-fine interface sources)
    int32_t ngh = 0;
    int32_t* gpb = nullptr;       // per ghost block: the 8 parent blocks around it, or -1
    uint32_t* ggroup = nullptr;   // group and pair words of the chunks (lb_kernels.h)
    uint32_t* gpair = nullptr;
    lbk::GhostChunk* gchunk = nullptr;
    int32_t pd[3] = {0, 0, 0};
    std::vector<int32_t> grid_host;  // host copy of grid, for the child level's ghost parents
    // Bouzidi link list
    int64_t nlinks = 0;
    // BouzidiLink<uint32_t> (lidx32, a population buffer below 2^32 slots) or
    // <uint64_t>, and the work entries' (first link, number of links)
    void* llink = nullptr;
    bool lidx32 = false;
    float* ltmp = nullptr;
    std::vector<std::pair<int32_t, int32_t>> lchunks;
    bool wide = false;    // population buffer >= 4 GiB: kernels use 64-bit offsets
    bool wide_g = false;  // the same for the thermal populations
    // work lists over this level alone (LevelArgs index = level index):
    // blocks in processing order, ghost-fill chunks, Bouzidi-link chunks
    lbk::Work* wcol = nullptr;
    int32_t n_gchunks = 0;
    lbk::Work* wgh = nullptr;
    int32_t n_lchunks = 0;
    lbk::Work* wlk = nullptr;
    int cur = 0;        // buffer index written by the last step (0 before any step)
    std::vector<int32_t> order_host;  // processing order (engine work lists)
    // Device block i holds the caller's block perm[i] (0-based); the device
    // order is the slab order of lb_level_upload.
    std::vector<int32_t> perm;
    int32_t n_int = 0;                // interior blocks: the first n_int of the order
    // kernel timing: event pairs recorded around collide launches
    // [0] stream-collide launches, [1] thermal launches
    std::vector<std::pair<hipEvent_t, hipEvent_t>> ev[2];
    size_t ev_used[2] = {0, 0};
};

}  // namespace

namespace {
// Whether a context's or engine's stream may hold steps that nobody has waited
// for: set before they are queued, cleared when the stream is found idle.
struct Queued {
    hipStream_t stream = nullptr;
    bool steps = false;  // under g_queued.mu
};
struct QueuedList {
    std::mutex mu;
    std::vector<Queued*> all;
};
QueuedList g_queued;

void queued_open(Queued* q, hipStream_t stream) {
    q->stream = stream;
    std::lock_guard<std::mutex> lk(g_queued.mu);
    g_queued.all.push_back(q);
}
void queued_close(Queued* q) {  // before the stream is destroyed
    std::lock_guard<std::mutex> lk(g_queued.mu);
    g_queued.all.erase(std::remove(g_queued.all.begin(), g_queued.all.end(), q), g_queued.all.end());
}
void queued_steps(Queued* q) {
    std::lock_guard<std::mutex> lk(g_queued.mu);
    q->steps = true;
}
// (self's stream has been waited for)
bool others_queued(Queued* self) {
    std::lock_guard<std::mutex> lk(g_queued.mu);
    self->steps = false;
    for (Queued* q : g_queued.all) {
        if (q == self || !q->steps) continue;
        if (hipStreamQuery(q->stream) != hipSuccess) {
            (void)hipGetLastError();  // "not ready" is no error of the launches that follow
            return true;
        }
        q->steps = false;
    }
    return false;
}
}  // namespace

struct lb_ctx {
    Queued queued;
    int device = 0;
    lb_config cfg{};
    hipStream_t stream = nullptr;
    const Kern* k = &kStrict;
    std::vector<Level> levels;
    std::vector<void*> allocs;
    int64_t bytes = 0;
    std::string err;
    // mesh
    int64_t n_tri = 0;
    float* mesh[7] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    float* maps[4] = {nullptr, nullptr, nullptr, nullptr};
    double* fpart = nullptr;
    double* spart = nullptr;
    int n_stat_groups = 0;
    // divergence check: one entry per level and a counter (allocated at creation)
    lbk::FiniteEntry* fin_ents = nullptr;
    int32_t* fin_count = nullptr;
    bool profile = false;
    // device-resident kernel arguments: the case record and one LevelArgs per level
    lbk::CaseState* st_dev = nullptr;
    lbk::LevelArgs* las_dev = nullptr;
    std::vector<lbk::LevelArgs> las_host;
    lb_engine* engine = nullptr;  // set while attached to a batched engine
    bool dry = false;             // footprint planning: nothing is allocated or copied
    bool counted = false;         // holds a share of the download pieces
};

// One attached case of an engine.
struct EngineCase {
    lb_ctx* c = nullptr;
    int64_t n_total = 0;
    int64_t t0 = 1;          // next coarse step (host copy of the device record)
    int32_t t_inc = 1;
    int32_t batch = 8;
    float* u_tab = nullptr;  // device, owned by the case context
    lb_step_params p{};
    // force sampling inside the engine step (lb_engine_sample_forces)
    double* acc = nullptr;   // device [10], owned by the case context
    bool sample = false;
    int64_t diag = 0, ramp = 0;
    lb_force_params fp{};
};

// Work lists of one depth of the engine's recursion (concatenated over cases).
struct DepthWork {
    lbk::Work *col = nullptr, *gh = nullptr, *lk = nullptr, *tcol = nullptr;
    int32_t ncol = 0, ngh = 0, nlk = 0, ntcol = 0;
    int wide = 0, wide_g = 0;
    // force sampling of the cases whose first level runs at this depth:
    // triangle chunks (li = record, item = chunk) and the record indices
    lbk::Work* fw = nullptr;
    int32_t* frec = nullptr;
    int32_t nfw = 0, nfrec = 0;
};

struct lb_engine {
    Queued queued;
    int device = 0;
    int32_t storage = 0;
    const Kern* k = &kStrict;
    hipStream_t stream = nullptr;
    std::vector<EngineCase> cases;
    std::string err;
    // batched launch data, rebuilt when the case set changes
    bool dirty = true;
    int lmax = 0;
    std::vector<void*> allocs;
    lbk::LevelArgs* las = nullptr;
    lbk::CaseState* states = nullptr;  // one record per attached case, contiguous
    lbk::EngineForce* frecs = nullptr; // force-sampling records
    std::vector<DepthWork> depth;
    int32_t n_active = 0;
    // options
    bool use_graph = true;
    int sched = LB_SCHED_LINEAR;
    int waves = 5;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    // divergence check buffers (grown on demand, kept across rebuilds)
    lbk::FiniteEntry* fin_ents = nullptr;
    int32_t* fin_counts = nullptr;
    size_t fin_cap_ents = 0, fin_cap_cases = 0;
};

namespace {

int fail(lb_ctx* c, int code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    std::vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    if (c) c->err = buf;
    return code;
}

#define HIPCHK(ctx, expr)                                                                                 \
    do {                                                                                                  \
        hipError_t e_ = (expr);                                                                           \
        if (e_ != hipSuccess) return fail(ctx, LB_EHIP, "%s: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__); \
    } while (0)

// Case buffers come from the device's default memory pool, allocated and
// freed in the order of the case's stream: a finished case's buffers go back
// to the pool without the device-wide wait and unmapping of hipFree (about
// 16 ms for the ~100 buffers of a case), and later cases reuse them.  The
// pool keeps up to 64 GiB of freed memory.
void setup_pool(int dev) {
    static std::atomic<bool> done[64];
    if (dev < 0 || dev >= 64 || done[dev].exchange(true)) return;
    hipMemPool_t pool;
    if (hipDeviceGetDefaultMemPool(&pool, dev) == hipSuccess) {
        uint64_t keep = 64ull << 30;
        (void)hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep);
    }
}

template <class T>
int dalloc(lb_ctx* c, T** p, size_t n) {
    *p = nullptr;
    size_t bytes = std::max<size_t>(n, 1) * sizeof(T);
    if (c->dry) {  // footprint planning: count only
        c->bytes += (int64_t)bytes;
        return LB_OK;
    }
    setup_pool(c->device);
    // usable from every stream once the case's stream has passed it
    hipError_t e = hipMallocAsync((void**)p, bytes, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) {
        *p = nullptr;
        (void)hipGetLastError();
        return fail(c, LB_ENOMEM, "hipMalloc(%zu bytes) failed: %s", bytes, hipGetErrorString(e));
    }
    c->allocs.push_back((void*)*p);
    c->bytes += (int64_t)bytes;
    return LB_OK;
}

template <class T>
int h2d(lb_ctx* c, T* dst, const T* src, size_t n) {
    if (c->dry) return LB_OK;
    hipError_t e = hipMemcpy(dst, src, n * sizeof(T), hipMemcpyHostToDevice);
    if (e != hipSuccess) return fail(c, LB_EHIP, "hipMemcpy H2D: %s", hipGetErrorString(e));
    return LB_OK;
}

// Counts what was allocated since `before` as `bytes` where that is more.  The
// byte count of a case is a result of the interface (lb_device_bytes,
// lb_footprint), which hosts record and compare, and does not follow the
// layout of the tables: one that got smaller goes on counting what it did.
// Nothing is allocated for the difference.
void count_as(lb_ctx* c, int64_t before, int64_t bytes) { c->bytes = std::max(c->bytes, before + bytes); }
// What a level's record counts.
constexpr int64_t kLevelRecord = 384;
static_assert((int64_t)sizeof(lbk::LevelArgs) <= kLevelRecord, "a case may not hold more than it counts");

float half_to_float(uint16_t h) {
    int s = (h >> 15) & 1, e = (h >> 10) & 31, m = h & 1023;
    float v;
    if (e == 0) v = std::ldexp((float)m, -24);
    else if (e == 31) v = m ? NAN : INFINITY;
    else v = std::ldexp((float)(m | 1024), e - 25);
    return s ? -v : v;
}

inline size_t fidx(int64_t b, int k, int c) { return ((size_t)b * Q + k) * NC + c; }

lbk::Work mkwork(int li, int item, int ci, const int32_t* row, int32_t flags = 0) {
    lbk::Work w;
    w.li = li;
    w.item = item;
    w.ci = ci;
    w.flags = flags;
    w.nbr_row = row;
    return w;
}

// Population storage on the host side of transfers.  FP16/BF16 levels hold
// f - w_k rounded to nearest even; the device decodes w_k + stored value.
float wk_host(int k) {
    const int cx = k % 3 - 1, cy = (k / 3) % 3 - 1, cz = k / 9 - 1;
    const int d2 = cx * cx + cy * cy + cz * cz;
    return d2 == 0 ? 8.0f / 27.0f : d2 == 1 ? 2.0f / 27.0f : d2 == 2 ? 1.0f / 54.0f : 1.0f / 216.0f;
}

size_t pop_bytes(int storage) { return storage == LB_STORAGE_FP32 ? 4 : 2; }

uint16_t float_to_half(float f) {
    uint32_t x;
    std::memcpy(&x, &f, 4);
    const uint32_t sign = (x >> 16) & 0x8000u, ax = x & 0x7fffffffu;
    if (ax > 0x7f800000u) return (uint16_t)(sign | 0x7e00u);
    if (ax >= 0x47800000u) return (uint16_t)(sign | 0x7c00u);  // |f| >= 65536 (and inf)
    if (ax < 0x38800000u) {                                      // half subnormal range: multiples of 2^-24
        const float v = std::nearbyint(std::fabs(f) * 16777216.0f);
        return (uint16_t)(sign | (uint32_t)v);
    }
    uint32_t h = ((((ax >> 23) - 112u) << 10) | ((ax >> 13) & 0x3ffu));
    const uint32_t rem = ax & 0x1fffu;
    if (rem > 0x1000u || (rem == 0x1000u && (h & 1u))) h++;  // carry into the exponent gives inf at 65520
    return (uint16_t)(sign | h);
}

uint16_t float_to_bf16(float f) {
    uint32_t b;
    std::memcpy(&b, &f, 4);
    if ((b & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((b >> 16) | 0x40u);
    b += 0x7fffu + ((b >> 16) & 1u);
    return (uint16_t)(b >> 16);
}

void encode_pop(uint8_t* base, size_t i, float f, int storage, float w) {
    if (storage == LB_STORAGE_FP32) {
        std::memcpy(base + i * 4, &f, 4);
        return;
    }
    const uint16_t u = storage == LB_STORAGE_FP16 ? float_to_half(f - w) : float_to_bf16(f - w);
    std::memcpy(base + i * 2, &u, 2);
}

#define RC(expr)                \
    do {                        \
        int rc_ = (expr);       \
        if (rc_ != LB_OK) return rc_; \
    } while (0)

// Build the Bouzidi link list of one level (src/geometry/bouzidi_kernel.jl:35-89):
// link (cell x, direction k) with q_min < q <= 1 corrects slot (x, opp k).
int build_links(lb_ctx* c, Level& L, const lb_level_desc* d) {
    const int64_t nbc = d->n_boundary_cells;
    if (nbc <= 0) return LB_OK;
    if (!d->bouzidi_cell_block || !d->bouzidi_cell_x || !d->bouzidi_cell_y || !d->bouzidi_cell_z ||
        (!d->bouzidi_q_dense && !d->bouzidi_q_cells))
        return fail(c, LB_EINVAL, "level %d: Bouzidi cell list or q map missing", d->level_id);
    const float qmin = c->cfg.q_min_threshold;
    const int64_t nb = d->n_blocks;
    std::vector<int64_t> dst, s1, s2;
    std::vector<float> ca, cb;
    for (int64_t i = 0; i < nbc; i++) {
        int b = d->bouzidi_cell_block[i], x = d->bouzidi_cell_x[i], y = d->bouzidi_cell_y[i],
            z = d->bouzidi_cell_z[i];
        if (b < 1 || b > nb || x < 1 || x > 8 || y < 1 || y > 8 || z < 1 || z > 8)
            return fail(c, LB_EINVAL, "level %d: Bouzidi cell %lld out of range", d->level_id, (long long)i);
        int cl = (x - 1) + 8 * (y - 1) + 64 * (z - 1);
        for (int k = 0; k < Q; k++) {
            // the dense q map is in the caller's block order
            const size_t bref = L.perm.empty() ? (size_t)(b - 1) : (size_t)L.perm[(size_t)b - 1];
            uint16_t bits = d->bouzidi_q_cells ? d->bouzidi_q_cells[i * Q + k]
                                               : d->bouzidi_q_dense[(size_t)cl + 512 * bref + 512 * (size_t)nb * k];
            float q = half_to_float(bits);
            if (!(q > qmin && q <= 1.0f)) continue;
            int ok = 26 - k;
            int cx = k % 3 - 1, cy = (k / 3) % 3 - 1, cz = k / 9 - 1;
            int64_t sA = (int64_t)fidx(b - 1, k, cl);
            int64_t sB;
            float a, bb;
            if (q < 0.5f) {
                int nx = x - cx, ny = y - cy, nz = z - cz;
                if (nx >= 1 && nx <= 8 && ny >= 1 && ny <= 8 && nz >= 1 && nz <= 8) {
                    sB = (int64_t)fidx(b - 1, k, (nx - 1) + 8 * (ny - 1) + 64 * (nz - 1));
                } else {
                    int ox = nx < 1 ? -1 : (nx > 8 ? 1 : 0), oy = ny < 1 ? -1 : (ny > 8 ? 1 : 0),
                        oz = nz < 1 ? -1 : (nz > 8 ? 1 : 0);
                    int dir = (ox + 1) + 3 * (oy + 1) + 9 * (oz + 1);
                    int nbb = d->neighbor_table[(size_t)(b - 1) + (size_t)nb * dir];
                    if (nbb > 0) {
                        int wx = nx < 1 ? nx + 8 : (nx > 8 ? nx - 8 : nx);
                        int wy = ny < 1 ? ny + 8 : (ny > 8 ? ny - 8 : ny);
                        int wz = nz < 1 ? nz + 8 : (nz > 8 ? nz - 8 : nz);
                        sB = (int64_t)fidx(nbb - 1, k, (wx - 1) + 8 * (wy - 1) + 64 * (wz - 1));
                    } else {
                        sB = sA;
                    }
                }
                float c1 = 2.0f * q;
                a = c1;
                bb = 1.0f - c1;
            } else {
                sB = (int64_t)fidx(b - 1, ok, cl);
                float t2 = 2.0f * q;
                float inv = 1.0f / t2;
                a = inv;
                bb = (2.0f * q - 1.0f) * inv;
            }
            dst.push_back((int64_t)fidx(b - 1, ok, cl));
            s1.push_back(sA);
            s2.push_back(sB);
            ca.push_back(a);
            cb.push_back(bb);
        }
    }
    L.nlinks = 0;
    if (dst.empty()) return LB_OK;
    if (dst.size() > (size_t)INT32_MAX) return fail(c, LB_EINVAL, "level %d: %zu wall links", d->level_id, dst.size());
    // One link per corrected slot.  A cell listed more than once gives the same
    // slots again; the last listing counts, as in a loop over the list that
    // reads the uncorrected populations.  (Two links of one slot could stand
    // in different work entries, and for q >= 0.5 the slot is its own second
    // source: whichever entry came later would correct the corrected value.)
    std::vector<std::pair<int64_t, int32_t>> listed(dst.size());  // slot, minus the place in the list
    for (size_t i = 0; i < dst.size(); i++) listed[i] = {dst[i], -(int32_t)i};
    std::sort(listed.begin(), listed.end());
    std::vector<int32_t> by_dst;
    by_dst.reserve(listed.size());
    for (size_t i = 0; i < listed.size(); i++)
        if (i == 0 || listed[i].first != listed[i - 1].first) by_dst.push_back(-listed[i].second);
    const size_t n = by_dst.size();
    L.nlinks = (int64_t)n;
    // Link order.  Sorted by destination, a wave's links share (block,
    // direction) rows, so its loads and stores of the same row coalesce.  A
    // work entry gathers its links' values before it stores any, so a link that
    // reads a slot which another link corrects (a cell with walls on both
    // sides, or two cells apart from one) has to be in the same entry: linked
    // links stand together, and entries of up to 256 links are cut between
    // such groups (one longer group makes one longer entry).
    std::vector<int32_t> group(n);
    for (size_t r = 0; r < n; r++) group[r] = (int32_t)r;  // over ranks in by_dst; the root is the lowest rank
    auto root = [&](int32_t r) {
        while (group[(size_t)r] != r) r = group[(size_t)r] = group[(size_t)group[(size_t)r]];
        return r;
    };
    // corrected slots as bits, per block that has any: few reads meet one
    std::vector<int32_t> block_row((size_t)nb, -1);
    std::vector<uint64_t> bits;
    constexpr size_t kRow = (size_t)Q * NC / 64;
    for (const int32_t i : by_dst) {
        const size_t blk = (size_t)dst[(size_t)i] / (Q * NC), at = (size_t)dst[(size_t)i] % (Q * NC);
        if (block_row[blk] < 0) {
            block_row[blk] = (int32_t)(bits.size() / kRow);
            bits.resize(bits.size() + kRow, 0);
        }
        bits[(size_t)block_row[blk] * kRow + at / 64] |= 1ull << (at % 64);
    }
    auto corrected = [&](int64_t slot) {
        const size_t blk = (size_t)slot / (Q * NC), at = (size_t)slot % (Q * NC);
        return block_row[blk] >= 0 && ((bits[(size_t)block_row[blk] * kRow + at / 64] >> (at % 64)) & 1u) != 0;
    };
    for (size_t r = 0; r < n; r++) {
        const size_t i = (size_t)by_dst[r];
        for (const int64_t slot : {s1[i], s2[i]}) {
            if (slot == dst[i] || !corrected(slot)) continue;
            const auto it = std::lower_bound(by_dst.begin(), by_dst.end(), slot,
                                             [&](int32_t u, int64_t v) { return dst[(size_t)u] < v; });
            if (it == by_dst.end() || dst[(size_t)*it] != slot) continue;
            const int32_t a = root((int32_t)r), b = root((int32_t)(it - by_dst.begin()));
            group[(size_t)std::max(a, b)] = std::min(a, b);
        }
    }
    std::unordered_map<int32_t, std::vector<int32_t>> members;  // groups of more than one link
    for (size_t r = 0; r < n; r++) {
        const int32_t g = root((int32_t)r);
        if (g != (int32_t)r) members[g].push_back((int32_t)r);
    }
    std::vector<int32_t> order;  // ranks, group by group
    order.reserve(n);
    L.lchunks.clear();
    int32_t first = 0;
    for (size_t r = 0; r < n; r++) {
        if (group[r] != (int32_t)r) continue;  // listed with its group
        const auto it = members.find((int32_t)r);
        const int32_t size = 1 + (it == members.end() ? 0 : (int32_t)it->second.size());
        const int32_t have = (int32_t)order.size() - first;
        if (have > 0 && have + size > 256) {
            L.lchunks.emplace_back(first, have);
            first = (int32_t)order.size();
        }
        order.push_back((int32_t)r);
        if (it != members.end()) order.insert(order.end(), it->second.begin(), it->second.end());
    }
    L.lchunks.emplace_back(first, (int32_t)order.size() - first);
    // 32-bit slots where the level's population buffer (ghost blocks and
    // padding included) has fewer than 2^32 of them.  wide_offsets keeps
    // 64-bit slots too.
    const uint64_t slots = ((uint64_t)nb + (uint64_t)L.ngh) * NC * Q + 512;
    L.lidx32 = c->cfg.wide_offsets == 0 && slots < ((uint64_t)1 << 32);
    auto upload_links = [&](auto zero) -> int {
        typedef decltype(zero) SlotT;
        std::vector<lbk::BouzidiLink<SlotT>> v(n);
        for (size_t q = 0; q < n; q++) {
            const size_t i = (size_t)by_dst[(size_t)order[q]];
            v[q] = {(SlotT)dst[i], (SlotT)s2[i], ca[i], cb[i]};
        }
        lbk::BouzidiLink<SlotT>* p = nullptr;
        RC(dalloc(c, &p, n));
        L.llink = p;
        return h2d(c, p, v.data(), n);
    };
    if (L.lidx32) RC(upload_links((uint32_t)0));
    else RC(upload_links((uint64_t)0));
    bool longer = false;
    for (const auto& e : L.lchunks) longer = longer || e.second > 256;
    if (longer) RC(dalloc(c, &L.ltmp, n));
    return LB_OK;
}

// perform_timestep_v2! + recursive_step! for one level (timestep.jl:1-159,
// solver_control.jl:6-197): substep j of level li counted from the coarse step
// t0 of the case record (t_sub = t0 * 2^li + j), then both child substeps.  The
// kernels resolve buffers, parity, seed and temporal weight from (record, j).
// Kernel timing: record the start event of kernel kind `which` (0 collide,
// 1 thermal) and hand back the end event to record after the launch.
int profile_begin(lb_ctx* c, Level& L, int which, hipEvent_t* end) {
    *end = nullptr;
    if (!c->profile) return LB_OK;
    auto& ev = L.ev[which];
    size_t& used = L.ev_used[which];
    if (used == ev.size()) {
        hipEvent_t x, y;
        HIPCHK(c, hipEventCreate(&x));
        HIPCHK(c, hipEventCreate(&y));
        ev.emplace_back(x, y);
    }
    HIPCHK(c, hipEventRecord(ev[used].first, c->stream));
    *end = ev[used].second;
    used++;
    return LB_OK;
}

// Occupancy of the stream-collide kernel per population storage: 6 waves per
// SIMD for 16-bit storage (launches of up to 1,280 blocks take 5 all the same,
// SMALL_TILES in lb_kernels.hip), 5 for FP32.  Measured through the engine, 5
// and 6 waves: FP16 1,434 and 1,428 us a coarse step (6.1 M cells), 2,389 and
// 2,425 (11.4 M, where interior and boundary blocks apart had 2,646 and 2,585),
// 4,503 and 4,501 (10.7 M, thermal); FP32 1,957 and 2,046 (6.1 M).
int default_waves(int storage) { return storage == LB_STORAGE_FP32 ? 5 : 6; }

int step_level(lb_ctx* c, int li, int64_t j) {
    if (li >= (int)c->levels.size()) return LB_OK;
    Level& L = c->levels[(size_t)li];
    const bool ddf = c->cfg.ddf_enabled && L.g[0] != nullptr;
    const int storage = c->cfg.storage;
    const lbk::LevelArgs* las = c->las_dev;
    const lbk::CaseState* st = c->st_dev;
    if (L.nb > 0) {
        // one ghost pass per parent step fills the inputs of both child substeps
        const bool fill = li > 0 && L.n_gchunks > 0 && (j & 1) == 0;
        if (fill) HIPCHK(c, c->k->ghost_fill(las, st, L.wgh, L.n_gchunks, j, storage, c->stream));
        hipEvent_t e1 = nullptr;
        RC(profile_begin(c, L, 0, &e1));
        HIPCHK(c, c->k->collide(las, st, L.wcol, L.nb, j, storage, L.wide ? 1 : 0, LB_SCHED_LINEAR,
                                default_waves(storage), c->stream));
        if (e1) HIPCHK(c, hipEventRecord(e1, c->stream));
        if (ddf) {
            hipEvent_t e2 = nullptr;
            RC(profile_begin(c, L, 1, &e2));
            HIPCHK(c, c->k->thermal(las, st, L.wcol, L.nb, j, storage, L.wide_g ? 1 : 0, LB_SCHED_LINEAR, c->stream));
            if (e2) HIPCHK(c, hipEventRecord(e2, c->stream));
        }
        if (L.n_lchunks > 0) HIPCHK(c, c->k->bouzidi(las, st, L.wlk, L.n_lchunks, j, storage, c->stream));
    }
    RC(step_level(c, li + 1, 2 * j));
    RC(step_level(c, li + 1, 2 * j + 1));
    return LB_OK;
}

// The case record for coarse step t with the given inlet velocity and the
// physics parameters of one lb_step_batch call.
lbk::CaseState case_record(int64_t t, float u, const lb_step_params* p, const lb_config& cfg) {
    lbk::CaseState s;
    std::memset(&s, 0, sizeof s);
    s.t0 = t;
    s.n_total = INT64_MAX;
    s.u = u;
    s.active = 1;
    s.t_inc = 1;
    s.batch = 1;
    s.u_tab = nullptr;
    s.c_wale = p->c_wale;
    s.nu_sgs_bg = p->nu_sgs_background;
    s.inlet_turb = p->inlet_turbulence;
    s.omega_bulk = p->omega_bulk;
    s.omega3 = p->omega_3;
    s.omega4 = p->omega_4;
    s.lambda = p->lambda_param;
    s.adaptive = p->adaptive_omega4;
    s.limiter = p->limiter;
    s.comp = p->compressible;
    s.wall_model = p->wall_model ? 1 : 0;
    s.sponge_blend = p->sponge_blend_distributions;
    s.T_inlet = p->T_inlet;
    s.T_wall = p->T_wall;
    s.adiabatic = p->wall_bc_adiabatic;
    s.temporal = cfg.temporal_interpolation ? 1 : 0;
    return s;
}

// Output half of every level after coarse step t: the last substep of level
// li is t * 2^li + 2^li - 1.
void set_current(lb_ctx* c, int64_t t) {
    for (size_t li = 0; li < c->levels.size(); li++) {
        const int64_t last = (t << li) + ((int64_t)1 << li) - 1;
        c->levels[li].cur = 1 - (int)(last & 1);
    }
}

// Work list of a level's wall links.
int link_list(lb_ctx* c, int li, Level& L) {
    L.n_lchunks = L.nlinks > 0 ? (int32_t)L.lchunks.size() : 0;
    if (L.n_lchunks == 0) return LB_OK;
    std::vector<lbk::Work> w;
    for (const auto& e : L.lchunks) w.push_back(mkwork(li, e.first, 0, nullptr, e.second));
    RC(dalloc(c, &L.wlk, w.size()));
    return h2d(c, L.wlk, w.data(), w.size());
}

// Work list of a level's ghost-fill chunks.
int ghost_list(lb_ctx* c, int li, Level& L) {
    if (L.n_gchunks == 0) return LB_OK;
    std::vector<lbk::Work> w((size_t)L.n_gchunks);
    for (int32_t i = 0; i < L.n_gchunks; i++) w[(size_t)i] = mkwork(li, i, 0, (const int32_t*)(L.gchunk + i));
    RC(dalloc(c, &L.wgh, w.size()));
    return h2d(c, L.wgh, w.data(), w.size());
}

// LevelArgs of level li (host copy + device record); the parent's pairs come
// from level li - 1, which is uploaded first.
int upload_level_args(lb_ctx* c, int li) {
    const Level& L = c->levels[(size_t)li];
    lbk::LevelArgs& A = c->las_host[(size_t)li];
    std::memset((void*)&A, 0, sizeof A);
    for (int i = 0; i < 2; i++) {
        A.f[i] = L.f[i];
        A.rho[i] = L.rho[i];
        A.vel[i] = L.vel[i];
        A.g[i] = L.g[i];
        A.T[i] = L.T[i];
    }
    A.obst = L.obst;
    A.sponge = L.sponge;
    A.wall_dist = L.wall_dist;
    A.nbr = L.nbr;
    A.borg = L.borg;
    A.nb = L.nb;
    const int scale = 1 << (L.id - 1);
    A.nxg = c->cfg.domain_nx * scale;
    A.nyg = c->cfg.domain_ny * scale;
    A.nzg = c->cfg.domain_nz * scale;
    A.lshift = L.id - 1;
    A.leaf = li + 1 == (int)c->levels.size() ? 1 : 0;
    A.tau = L.tau;
    A.tau_g = L.tau_g;
    if (li > 0) {
        const Level& P = c->levels[(size_t)li - 1];
        // The ghost fill reads block 0 of the parent in place of a corner that
        // the parent level does not hold, and drops what it read.  A parent
        // without blocks has no block 0 to read; the level's own stands in.
        const Level& S = P.nb > 0 ? P : L;
        for (int i = 0; i < 2; i++) {
            A.pf[i] = S.f[i];
            A.prho[i] = S.rho[i];
            A.pvel[i] = S.vel[i];
            A.pg[i] = S.g[i];
            A.pT[i] = S.T[i];
        }
        A.ptau = P.tau;
        A.ptau_g = P.tau_g;
    }
    A.gpb = L.gpb;
    A.ggroup = L.ggroup;
    A.gpair = L.gpair;
    A.links.n = L.nlinks;
    A.links.link = L.llink;
    A.links.tmp = L.ltmp;
    A.links.idx32 = L.lidx32 ? 1 : 0;
    return h2d(c, c->las_dev + li, &A, 1);
}

int efail(lb_engine* e, int code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    std::vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    if (e) e->err = buf;
    return code;
}

#define EHIPCHK(eng, expr)                                                                                \
    do {                                                                                                  \
        hipError_t e_ = (expr);                                                                           \
        if (e_ != hipSuccess) return efail(eng, LB_EHIP, "%s: %s", #expr, hipGetErrorString(e_));        \
    } while (0)

void engine_free_lists(lb_engine* e) {
    if (e->exec) (void)hipGraphExecDestroy(e->exec);
    if (e->graph) (void)hipGraphDestroy(e->graph);
    e->exec = nullptr;
    e->graph = nullptr;
    for (void* p : e->allocs) (void)hipFree(p);
    e->allocs.clear();
    e->las = nullptr;
    e->states = nullptr;
    e->frecs = nullptr;
    e->depth.clear();
}

template <class T>
int eupload(lb_engine* e, T** dst, const std::vector<T>& v) {
    *dst = nullptr;
    if (v.empty()) return LB_OK;
    EHIPCHK(e, hipMalloc((void**)dst, v.size() * sizeof(T)));
    e->allocs.push_back((void*)*dst);
    EHIPCHK(e, hipMemcpy(*dst, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return LB_OK;
}

lbk::ForceArgs force_args(lb_ctx* c, const lb_force_params* fp, float side);

// The device record of an attached case at its current position.
lbk::CaseState engine_record(const lb_engine* e, const EngineCase& ec) {
    lbk::CaseState r = case_record(ec.t0, 0.0f, &ec.p, ec.c->cfg);
    r.n_total = ec.n_total;
    r.active = ec.t0 <= ec.n_total ? 1 : 0;
    r.t_inc = ec.t_inc;
    r.batch = ec.batch;
    r.u_tab = ec.u_tab;
    (void)e;
    return r;
}

// Rebuild the concatenated LevelArgs, the per-depth work lists and the case
// records after the case set changed.  Cases are aligned on their finest
// level: level l of a case with L levels runs at depth l + (Lmax - L).
int engine_rebuild(lb_engine* e) {
    EHIPCHK(e, hipStreamSynchronize(e->stream));
    engine_free_lists(e);
    e->lmax = 0;
    for (const EngineCase& ec : e->cases) e->lmax = std::max(e->lmax, (int)ec.c->levels.size());
    std::vector<lbk::LevelArgs> las;
    std::vector<lbk::CaseState> sts;
    std::vector<int> base;
    for (EngineCase& ec : e->cases) {
        base.push_back((int)las.size());
        for (const lbk::LevelArgs& a : ec.c->las_host) las.push_back(a);
        ec.t_inc = 1 << (e->lmax - (int)ec.c->levels.size());
        sts.push_back(engine_record(e, ec));
    }
    RC(eupload(e, &e->las, las));
    RC(eupload(e, &e->states, sts));
    // force sampling: one record per sampling case, its triangle chunks
    // listed at the depth of the case's first level
    std::vector<lbk::EngineForce> frecs;
    std::vector<std::vector<lbk::Work>> fw((size_t)e->lmax);
    std::vector<std::vector<int32_t>> frec((size_t)e->lmax);
    for (size_t i = 0; i < e->cases.size(); i++) {
        EngineCase& ec = e->cases[i];
        if (!ec.sample) continue;
        lb_ctx* c = ec.c;
        const Level& fin = c->levels.back();
        lbk::EngineForce r;
        std::memset((void*)&r, 0, sizeof r);
        r.a = force_args(c, &ec.fp, 1.0f);
        r.rho2[0] = fin.rho[0];
        r.rho2[1] = fin.rho[1];
        r.diag = ec.diag;
        r.ramp = ec.ramp;
        r.ci = (int32_t)i;
        r.leaf_shift = (int32_t)c->levels.size() - 1;
        r.n_groups = (int32_t)((c->n_tri + 255) / 256);
        r.acc = ec.acc;
        const int d = e->lmax - (int)c->levels.size() + 1;
        const int32_t ri = (int32_t)frecs.size();
        for (int32_t g = 0; g < r.n_groups; g++) fw[(size_t)d - 1].push_back(mkwork(ri, g, (int32_t)i, nullptr));
        frec[(size_t)d - 1].push_back(ri);
        frecs.push_back(r);
    }
    RC(eupload(e, &e->frecs, frecs));
    e->depth.assign((size_t)e->lmax, DepthWork());
    for (int d = 1; d <= e->lmax; d++) {
        DepthWork& W = e->depth[(size_t)d - 1];
        RC(eupload(e, &W.fw, fw[(size_t)d - 1]));
        RC(eupload(e, &W.frec, frec[(size_t)d - 1]));
        W.nfw = (int32_t)fw[(size_t)d - 1].size();
        W.nfrec = (int32_t)frec[(size_t)d - 1].size();
    }
    for (int d = 1; d <= e->lmax; d++) {
        std::vector<lbk::Work> col, colb, gh, lk, tcol, tcolb;  // colb, tcolb: boundary blocks, listed last
        DepthWork& W = e->depth[(size_t)d - 1];
        for (size_t i = 0; i < e->cases.size(); i++) {
            const lb_ctx* c = e->cases[i].c;
            const int L = (int)c->levels.size();
            const int l = d - (e->lmax - L);
            if (l < 1 || l > L) continue;
            const Level& lev = c->levels[(size_t)l - 1];
            const int li = base[i] + l - 1, ci = (int)i;
            if (lev.nb == 0) continue;
            const bool ddf = c->cfg.ddf_enabled && lev.g[0] != nullptr;
            for (size_t q = 0; q < lev.order_host.size(); q++) {
                const int32_t b = lev.order_host[q];
                const bool interior = (int32_t)q < lev.n_int;
                const lbk::Work w = mkwork(li, b, ci, lev.nbr + (size_t)b * Q, lev.wflags[(size_t)b]);
                (interior ? col : colb).push_back(w);
                if (ddf) (interior ? tcol : tcolb).push_back(w);
            }
            for (int32_t q = 0; q < lev.n_gchunks; q++) gh.push_back(mkwork(li, q, ci, (const int32_t*)(lev.gchunk + q)));
            for (const auto& ch : lev.lchunks) lk.push_back(mkwork(li, ch.first, ci, nullptr, ch.second));
            if (lev.wide) W.wide = 1;
            if (lev.wide_g) W.wide_g = 1;
        }
        col.insert(col.end(), colb.begin(), colb.end());
        tcol.insert(tcol.end(), tcolb.begin(), tcolb.end());
        RC(eupload(e, &W.col, col));
        RC(eupload(e, &W.gh, gh));
        RC(eupload(e, &W.lk, lk));
        RC(eupload(e, &W.tcol, tcol));
        W.ncol = (int32_t)col.size();
        W.ngh = (int32_t)gh.size();
        W.nlk = (int32_t)lk.size();
        W.ntcol = (int32_t)tcol.size();
    }
    e->n_active = (int32_t)e->cases.size();
    e->dirty = false;
    return LB_OK;
}

// One depth-d operation (substep j) and its subtree, over all cases.
hipError_t engine_op(lb_engine* e, int d, int64_t j) {
    const DepthWork& W = e->depth[(size_t)d - 1];
    const Kern* k = e->k;
    hipError_t r = hipSuccess;
#define ETRY(x)                       \
    do {                              \
        r = (x);                      \
        if (r != hipSuccess) return r; \
    } while (0)
    const lbk::CaseState* st = e->states;
    // one ghost pass per parent step fills the inputs of both child substeps
    const bool fill = (j & 1) == 0;
    if (W.ngh && fill) ETRY(k->ghost_fill(e->las, st, W.gh, W.ngh, j, e->storage, e->stream));
    if (W.ncol)
        ETRY(k->collide(e->las, st, W.col, W.ncol, j, e->storage, W.wide, e->sched, e->waves, e->stream));
    if (W.ntcol) {
        // the thermal kernel has no persistent form
        const int tsched = e->sched == LB_SCHED_PERSISTENT ? LB_SCHED_LINEAR : e->sched;
        ETRY(k->thermal(e->las, st, W.tcol, W.ntcol, j, e->storage, W.wide_g, tsched, e->stream));
    }
    if (W.nlk) ETRY(k->bouzidi(e->las, st, W.lk, W.nlk, j, e->storage, e->stream));
    if (d < e->lmax) {
        ETRY(engine_op(e, d + 1, 2 * j));
        ETRY(engine_op(e, d + 1, 2 * j + 1));
    }
    // coarse step t0 + j of the cases whose first level runs at depth d is complete
    if (W.nfw) ETRY(k->engine_forces(e->frecs, st, W.fw, W.nfw, W.frec, W.nfrec, j, e->stream));
#undef ETRY
    return r;
}

hipError_t engine_issue_step(lb_engine* e) {
    hipError_t r = engine_op(e, 1, 0);
    if (r != hipSuccess) return r;
    return e->k->advance(e->states, (int32_t)e->cases.size(), e->stream);
}

// Divergence check entry of one level: its density and velocity in buffer
// `cur` (the output of the last completed coarse step).
int64_t largest(const std::vector<lbk::FiniteEntry>& ents) {  // cells of the largest entry
    int64_t n = 0;
    for (const lbk::FiniteEntry& e : ents) n = std::max(n, e.n);
    return n;
}
lbk::FiniteEntry finite_entry(const Level& L, int cur, int32_t slot) {
    lbk::FiniteEntry e;
    e.rho = L.rho[cur];
    e.vel = L.vel[cur];
    e.n = (int64_t)L.nb * NC;
    e.slot = slot;
    e.pad = 0;
    return e;
}

// The device buffers of lb_create.
int create_buffers(lb_ctx* c) {
    const size_t n = c->levels.size();
    RC(dalloc(c, &c->st_dev, 1));
    const int64_t before = c->bytes;
    RC(dalloc(c, &c->las_dev, n));
    count_as(c, before, (int64_t)n * kLevelRecord);
    RC(dalloc(c, &c->fin_ents, n));
    return dalloc(c, &c->fin_count, 1);
}

int check_ctx(lb_ctx* c) {
    if (!c) return LB_EINVAL;
    if (c->engine) return fail(c, LB_ESTATE, "case is attached to an engine");
    for (size_t i = 0; i < c->levels.size(); i++)
        if (!c->levels[i].uploaded) return fail(c, LB_ESTATE, "level %zu not uploaded", i + 1);
    return LB_OK;
}

}  // namespace

// ---------------------------------------------------------------------------
// lb_stats_noalloc: the statistics of lb_stats with their partial rows and
// the reduced result in a fixed device array instead of memory allocated on
// first use, for callers that cannot allocate.  One copy of the array per
// device; its address on each device is taken once, at context creation on
// that device (hipGetSymbolAddress), and only that address is handed to
// kernels and copies.
namespace {
constexpr int kStatsRows = 1024;  // the statistics kernel runs at most this many work-groups
constexpr size_t kScratchDoubles = (size_t)kStatsRows * 8 + 8;
constexpr int kMaxDevices = 64;
}  // namespace

static __device__ __align__(256) double scratch[kScratchDoubles];

namespace {
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};
hipError_t g_scratch_err[kMaxDevices] = {};

// Address of `scratch` on `device` (the current device), taken once.
void scratch_setup(int device) {
    if (device < 0 || device >= kMaxDevices) return;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[device]) return;
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e == hipSuccess && p) g_scratch_ptr[device] = (double*)p;
    else {
        g_scratch_err[device] = e;
        (void)hipGetLastError();
    }
}

double* scratch_on(int device, hipError_t* err) {
    if (device < 0 || device >= kMaxDevices) {
        *err = hipErrorInvalidDevice;
        return nullptr;
    }
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    *err = g_scratch_err[device];
    return g_scratch_ptr[device];
}

// The partial rows reduced in row order, with the operations lb_stats
// applies on the host (so the results are the same to the bit).
__global__ void stats_reduce_kernel(const double* __restrict__ part, int rows, double* __restrict__ out) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    double s0 = 0, s1 = 0, s4 = 0, s5 = 0, s6 = 0, mn = 1e300, mx = -1e300, vmax = 0;
    for (int g = 0; g < rows; g++) {
        const double* q = part + (size_t)g * 8;
        s0 += q[0];
        s1 += q[1];
        mn = q[2] < mn ? q[2] : mn;
        mx = mx < q[3] ? q[3] : mx;
        s4 += q[4];
        s5 += q[5];
        s6 += q[6];
        vmax = vmax < q[7] ? q[7] : vmax;
    }
    out[0] = s0; out[1] = s1; out[2] = mn; out[3] = mx;
    out[4] = s4; out[5] = s5; out[6] = s6; out[7] = vmax;
}
}  // namespace

// ---------------------------------------------------------------------------
// Field downloads.  A kernel puts a field's blocks in the caller's order,
// decodes it, and writes it into pinned host memory in pieces; threads copy
// the pieces to the caller's array as they arrive.  (A copy of the whole field
// into pageable memory and the permutation there by one thread ran at 3 to 5
// GB/s -- page faults of both arrays, then the copy -- against 18 GB/s now for
// 1.3 M cells and 44 GB/s for 52.5 M: velocity 4.4 -> 0.9 ms and 204 -> 14 ms.)
// While another context or an engine has steps queued, the pieces come over as
// copies of the blocks as they lie, and the threads reorder and decode them: a
// process has 4 hardware queues for all of its streams, so the kernel of an
// idle context may stand behind everything that a busy one has queued (260 ms
// behind 3,000 coarse steps of 1.3 M cells, for 2 of 16 contexts; as a copy
// 0.1 ms), and an event behind a copy would too.  Otherwise the kernel: copies
// need a quarter to a half longer for 6 to 52.5 M cells, and up to 0.1 ms more
// for each of the smallest (55 k cells).  Which one is settled as the download
// begins; steps that another thread queues meanwhile can still come before the
// kernel's next piece.
// The pinned memory is 8 pieces of 4 MiB for the process, allocated when first
// needed and given back with the last context.  A piece is held while it is
// filled and read, never while a context's earlier work is waited for, so
// downloads of different contexts run side by side; the pieces go round in the
// order of asking.  No piece is freed while a context lives: hipHostFree waits
// for everything queued on the device (340 ms behind 1,500 such steps, where
// hipHostMalloc takes 0.2 ms).
namespace {
constexpr size_t kPiece = (size_t)4 << 20;  // bytes; a multiple of a 512-float row
constexpr int kPieces = 8;

struct Piece {
    float* buf = nullptr;
    size_t bytes = 0;
    bool held = false;
};
struct Staging {
    std::mutex mu;  // held for these fields alone, not over a call to the device
    std::condition_variable cv;
    Piece piece[kPieces];
    uint64_t asked = 0, served = 0;
    int contexts = 0;
};
Staging g_staging;

void staging_context(int change) {
    float* spare[kPieces];
    int n = 0;
    {
        std::lock_guard<std::mutex> lk(g_staging.mu);
        g_staging.contexts += change;
        if (g_staging.contexts > 0) return;
        for (Piece& p : g_staging.piece) {
            if (p.held || !p.buf) continue;
            spare[n++] = p.buf;
            p.buf = nullptr;
            p.bytes = 0;
        }
    }
    for (int i = 0; i < n; i++) (void)hipHostFree(spare[i]);
}

// The next free piece, one that has its memory if there is any.
Piece* staging_take() {
    std::unique_lock<std::mutex> lk(g_staging.mu);
    const uint64_t turn = g_staging.asked++;
    Piece* p = nullptr;
    g_staging.cv.wait(lk, [&] {
        if (turn != g_staging.served) return false;
        for (Piece& q : g_staging.piece)
            if (!q.held && (!p || (!p->buf && q.buf))) p = &q;
        return p != nullptr;
    });
    p->held = true;
    g_staging.served++;
    lk.unlock();
    g_staging.cv.notify_all();
    return p;
}

void staging_give(Piece* p) {
    {
        std::lock_guard<std::mutex> lk(g_staging.mu);
        p->held = false;
    }
    g_staging.cv.notify_all();
}

// Memory for a piece in hand; less than a whole piece when memory is short.
hipError_t staging_fill(Piece* p) {
    hipError_t e = hipSuccess;
    for (size_t bytes = kPiece; !p->buf && bytes >= 65536; bytes /= 2) {
        e = hipHostMalloc((void**)&p->buf, bytes, hipHostMallocPortable);
        if (e == hipSuccess) {
            p->bytes = bytes;
        } else {
            p->buf = nullptr;
            (void)hipGetLastError();
        }
    }
    return p->buf ? hipSuccess : e;
}

// A row of 512 populations as the device stores it, decoded (lb_kernels.hip,
// Codec): w_k + the stored value.  FP16 without FP32 subnormals on the way, so
// that a thread's flush mode does not matter.
void decode_row(const uint8_t* src, int storage, float w, float* out) {
    if (storage == LB_STORAGE_FP32) {
        std::memcpy(out, src, (size_t)NC * 4);
        return;
    }
    uint16_t h[NC];
    std::memcpy(h, src, sizeof h);
    for (int i = 0; i < NC; i++) {
        uint32_t bits;
        if (storage == LB_STORAGE_BF16) {
            bits = (uint32_t)h[i] << 16;
        } else {
            const uint32_t a = (uint32_t)(h[i] & 0x7fffu) << 13, e = a & 0x0f800000u;
            // exponent 0: 2^-14 (1 + m) - 2^-14; 31: inf and NaN
            const float small = __builtin_bit_cast(float, a + 0x38800000u) - 6.103515625e-05f;
            const uint32_t b = e == 0u ? __builtin_bit_cast(uint32_t, small)
                                       : a + (e == 0x0f800000u ? 0x70000000u : 0x38000000u);
            bits = b | (uint32_t)(h[i] & 0x8000u) << 16;
        }
        out[i] = w + __builtin_bit_cast(float, bits);
    }
}

// Field `src` of n_comp components to dst (component k of the caller's block i
// at row k nb + i).  The context's stream is idle on entry.
int download_field(lb_ctx* c, const Level& L, const void* src, int n_comp, int storage, bool population, float* dst) {
    const int64_t nb = L.nb;
    if (nb == 0) return LB_OK;
    const bool copies = others_queued(&c->queued);
    const size_t row = (size_t)NC * pop_bytes(storage);
    // what a piece is filled with: device blocks, or rows of the caller's array
    const size_t unit = copies ? row * (size_t)n_comp : (size_t)NC * 4;
    const int64_t units = copies ? nb : nb * n_comp;
    const int workers = (int)std::min<uint64_t>(kPieces, ((uint64_t)units * unit + kPiece - 1) / kPiece);
    std::mutex launch;
    std::atomic<int64_t> next{0};  // first unit that no worker has
    std::atomic<int> err{(int)hipSuccess};
    // A worker takes a piece, has the next units put into it, and stores them.
    // All use the case's stream, so a piece is filled while the other workers
    // empty theirs.
    auto work = [&]() noexcept {
        hipEvent_t done = nullptr;
        hipError_t e = hipSetDevice(c->device);
        // (one worker: its launches are all that the stream holds)
        if (e == hipSuccess && workers > 1 && !copies) e = hipEventCreateWithFlags(&done, hipEventDisableTiming);
        while (e == hipSuccess && err.load() == (int)hipSuccess && next.load() < units) {
            Piece* const p = staging_take();
            e = staging_fill(p);
            const int64_t per = (int64_t)(p->bytes / unit), u0 = e == hipSuccess ? next.fetch_add(per) : units,
                          n = std::min(per, units - u0);
            if (n > 0 && copies) {
                e = hipMemcpyWithStream(p->buf, (const uint8_t*)src + (size_t)u0 * unit, (size_t)n * unit,
                                        hipMemcpyDeviceToHost, c->stream);
                for (int64_t b = 0; e == hipSuccess && b < n; b++)
                    for (int k = 0; k < n_comp; k++)
                        decode_row((const uint8_t*)p->buf + (size_t)b * unit + (size_t)k * row, storage,
                                   population ? wk_host(k) : 0.0f,
                                   dst + ((size_t)k * (size_t)nb + (size_t)L.perm[(size_t)(u0 + b)]) * NC);
            } else if (n > 0) {
                {
                    std::lock_guard<std::mutex> ll(launch);
                    e = c->k->export_rows(src, L.inv, L.nb, n_comp, storage, u0, (int32_t)n, p->buf, c->stream);
                    if (e == hipSuccess && done) e = hipEventRecord(done, c->stream);
                }
                if (e == hipSuccess) e = done ? hipEventSynchronize(done) : hipStreamSynchronize(c->stream);
                if (e == hipSuccess) std::memcpy(dst + (size_t)u0 * NC, p->buf, (size_t)n * unit);
            }
            if (e != hipSuccess) (void)hipStreamSynchronize(c->stream);  // nothing writes a piece once it is given back
            staging_give(p);
        }
        if (done) (void)hipEventDestroy(done);
        if (e != hipSuccess) err.store((int)e);
    };
    std::thread threads[kPieces - 1];
    for (int w = 0; w + 1 < workers; w++) {
        try {
            threads[w] = std::thread(work);
        } catch (...) {  // no thread to be had: the others take its share
        }
    }
    work();
    for (std::thread& t : threads)
        if (t.joinable()) t.join();
    const hipError_t e = (hipError_t)err.load();
    if (e != hipSuccess)
        return fail(c, e == hipErrorOutOfMemory ? LB_ENOMEM : LB_EHIP, "field download: %s", hipGetErrorString(e));
    return LB_OK;
}
}  // namespace

namespace lbsync {
CaptureLock& capture_mutex() {
    static CaptureLock m;
    return m;
}
}  // namespace lbsync

extern "C" {

const char* lb_last_error(const lb_ctx* ctx) { return ctx ? ctx->err.c_str() : "null context"; }

const char* lb_version(void) { return "ludwig_hip 0.1 gfx950"; }

int lb_create(lb_ctx** out, int device, const lb_config* cfg) {
    lbsync::SetupGuard guard;
    if (!out || !cfg) return LB_EINVAL;
    *out = nullptr;
    if (cfg->n_levels < 1 || cfg->n_levels > 16 || cfg->domain_nx < 8 || cfg->domain_ny < 8 || cfg->domain_nz < 8)
        return LB_EINVAL;
    if (cfg->storage != LB_STORAGE_FP32 && cfg->storage != LB_STORAGE_FP16 && cfg->storage != LB_STORAGE_BF16)
        return LB_EINVAL;
    lb_ctx* c = new lb_ctx();
    c->device = device;
    c->cfg = *cfg;
    c->k = cfg->strict_fp ? &kStrict : &kFast;
    hipError_t e = hipSetDevice(device);
    if (e != hipSuccess) {
        delete c;
        return LB_EHIP;
    }
    e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        delete c;
        return LB_EHIP;
    }
    scratch_setup(device);
    c->levels.resize((size_t)cfg->n_levels);
    c->las_host.resize((size_t)cfg->n_levels);
    std::memset((void*)c->las_host.data(), 0, c->las_host.size() * sizeof(lbk::LevelArgs));
    if (create_buffers(c) != LB_OK) {
        lb_destroy(c);
        return LB_ENOMEM;
    }
    queued_open(&c->queued, c->stream);
    staging_context(1);
    c->counted = true;
    *out = c;
    return LB_OK;
}

void lb_destroy(lb_ctx* c) {
    lbsync::SetupGuard guard;
    if (!c) return;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    for (auto& L : c->levels)
        for (auto& evk : L.ev)
            for (auto& e : evk) {
                (void)hipEventDestroy(e.first);
                (void)hipEventDestroy(e.second);
            }
    if (c->stream) {
        queued_close(&c->queued);
        for (void* p : c->allocs) (void)hipFreeAsync(p, c->stream);
        (void)hipStreamSynchronize(c->stream);
        (void)hipStreamDestroy(c->stream);
    }
    if (c->counted) staging_context(-1);
    delete c;
}

int lb_level_upload(lb_ctx* c, const lb_level_desc* d) {
    lbsync::SetupGuard guard;
    if (!c || !d) return LB_EINVAL;
    if (d->level_id < 1 || d->level_id > (int)c->levels.size())
        return fail(c, LB_EINVAL, "level_id %d out of range", d->level_id);
    Level& L = c->levels[(size_t)d->level_id - 1];
    if (L.uploaded) return fail(c, LB_ESTATE, "level %d already uploaded", d->level_id);
    if (d->level_id > 1 && !c->levels[(size_t)d->level_id - 2].uploaded)
        return fail(c, LB_ESTATE, "levels must be uploaded in order");
    const int32_t nb = d->n_blocks;
    if (nb < 0 || (nb > 0 && (!d->map_x || !d->map_y || !d->map_z || !d->neighbor_table || !d->obstacle ||
                             !d->sponge || !d->block_pointer)))
        return fail(c, LB_EINVAL, "level %d: missing arrays", d->level_id);
    if (d->ptr_dim_x < 0 || d->ptr_dim_y < 0 || d->ptr_dim_z < 0)
        return fail(c, LB_EINVAL, "level %d: bad block_pointer dims", d->level_id);
    if (!c->dry) HIPCHK(c, hipSetDevice(c->device));
    // Device block order.  The caller's blocks come in the reference's
    // lexicographic (bx, by, bz) order, z fastest.  On the device they are
    // stored, and processed, in 4-layer z-slabs: inside a slab x-rows of
    // 4-block z-columns, x fastest, then y.  The stream-collide pull reads a
    // 4-byte value per cell of each x face of a neighbour block out of
    // 128-byte lines that hold 4 rows of 8 cells (a y face reads one 32-byte
    // run per line, a z face whole lines), so x neighbours should be read
    // right after each other and y and z neighbours soon after, while their
    // lines are still in L2 or the last-level cache; and processing in
    // storage order streams the level through memory.  Measured on the
    // 52.5M-cell cube case (MI355X, FP32), finest stream-collide: the
    // caller's order with the slab work order dealt to XCDs in runs 1680 us;
    // slab storage in order 1545 us (1612 us in XCD runs); x fastest in order
    // 1904 us (the z neighbours fall out of the caches); the caller's order in
    // order 1634 us.  A 2-D Morton order of the columns in place of the
    // x-rows measured the same.  Every per-block input is permuted here and
    // every per-block output is permuted back (lb_download_level,
    // lb_upload_level); per-cell results do not depend on the order.
    std::vector<int32_t> perm((size_t)std::max(nb, 0)), inv((size_t)std::max(nb, 0));
    for (int32_t b = 0; b < nb; b++) perm[(size_t)b] = b;
    auto slab_key = [d](int32_t b) -> uint64_t {
        const uint64_t x = (uint64_t)(d->map_x[b] - 1), y = (uint64_t)(d->map_y[b] - 1), z = (uint64_t)(d->map_z[b] - 1);
        return ((z >> 2) << 48) | (y << 32) | (x << 8) | (z & 3u);
    };
    std::stable_sort(perm.begin(), perm.end(), [&slab_key](int32_t a, int32_t b) { return slab_key(a) < slab_key(b); });
    for (int32_t i = 0; i < nb; i++) inv[(size_t)perm[(size_t)i]] = i;
    std::vector<int32_t> pmx((size_t)std::max(nb, 0)), pmy(pmx.size()), pmz(pmx.size()), pnt((size_t)std::max(nb, 0) * Q);
    std::vector<uint8_t> pobst((size_t)std::max(nb, 0) * NC);
    std::vector<float> psponge(pobst.size()), pwall(d->wall_dist ? pobst.size() : 0);
    std::vector<int32_t> pbp((size_t)d->ptr_dim_x * d->ptr_dim_y * d->ptr_dim_z);
    std::vector<int32_t> pcell((size_t)std::max<int64_t>(d->n_boundary_cells, 0));
    lb_level_desc dp = *d;
    if (nb > 0) {
        for (int32_t i = 0; i < nb; i++) {
            const int32_t b = perm[(size_t)i];
            pmx[(size_t)i] = d->map_x[b];
            pmy[(size_t)i] = d->map_y[b];
            pmz[(size_t)i] = d->map_z[b];
            for (int k = 0; k < Q; k++) {
                const int v = d->neighbor_table[(size_t)b + (size_t)nb * k];
                pnt[(size_t)i + (size_t)nb * k] = (v >= 1 && v <= nb) ? inv[(size_t)v - 1] + 1 : v;
            }
            std::memcpy(&pobst[(size_t)i * NC], d->obstacle + (size_t)b * NC, NC);
            std::memcpy(&psponge[(size_t)i * NC], d->sponge + (size_t)b * NC, NC * sizeof(float));
            if (d->wall_dist) std::memcpy(&pwall[(size_t)i * NC], d->wall_dist + (size_t)b * NC, NC * sizeof(float));
        }
        for (size_t i = 0; i < pbp.size(); i++) {
            const int v = d->block_pointer[i];
            pbp[i] = (v >= 1 && v <= nb) ? inv[(size_t)v - 1] + 1 : v;
        }
        for (size_t i = 0; i < pcell.size() && d->bouzidi_cell_block; i++) {
            const int v = d->bouzidi_cell_block[i];
            pcell[i] = (v >= 1 && v <= nb) ? inv[(size_t)v - 1] + 1 : v;
        }
        dp.map_x = pmx.data();
        dp.map_y = pmy.data();
        dp.map_z = pmz.data();
        dp.neighbor_table = pnt.data();
        dp.block_pointer = pbp.empty() ? d->block_pointer : pbp.data();
        dp.obstacle = pobst.data();
        dp.sponge = psponge.data();
        dp.wall_dist = d->wall_dist ? pwall.data() : nullptr;
        if (d->bouzidi_cell_block) dp.bouzidi_cell_block = pcell.data();
    }
    L.perm = perm;
    d = &dp;
    L.id = d->level_id;
    L.nb = nb;
    L.tau = d->tau;
    L.tau_g = d->tau_g;
    L.dx = d->dx;
    // Host tables: 0-based neighbour rows, block origins, and ghost blocks for
    // in-domain neighbour positions the level does not hold (levels > 1).
    std::vector<int32_t> nbr((size_t)nb * Q), borg((size_t)nb * 3);
    const int scale = 1 << (L.id - 1);
    const int64_t dbx = (int64_t)c->cfg.domain_nx * scale / 8, dby = (int64_t)c->cfg.domain_ny * scale / 8,
                  dbz = (int64_t)c->cfg.domain_nz * scale / 8;
    auto key = [](int64_t x, int64_t y, int64_t z) { return (uint64_t)(x + 1) | ((uint64_t)(y + 1) << 21) | ((uint64_t)(z + 1) << 42); };
    std::unordered_map<uint64_t, int32_t> real, ghost;
    std::vector<int64_t> gpos;
    for (int32_t b = 0; b < nb; b++) real[key(d->map_x[b], d->map_y[b], d->map_z[b])] = b;
    for (int32_t b = 0; b < nb; b++) {
        for (int k = 0; k < Q; k++) {
            int v = d->neighbor_table[(size_t)b + (size_t)nb * k];
            if (v < 0 || v > nb) return fail(c, LB_EINVAL, "level %d: neighbour table entry out of range", L.id);
            int32_t id = v - 1;
            if (id < 0 && L.id > 1) {
                int64_t px = d->map_x[b] + k % 3 - 1, py = d->map_y[b] + (k / 3) % 3 - 1, pz = d->map_z[b] + k / 9 - 1;
                if (px >= 1 && px <= dbx && py >= 1 && py <= dby && pz >= 1 && pz <= dbz) {
                    auto it = ghost.find(key(px, py, pz));
                    if (it == ghost.end()) {
                        it = ghost.emplace(key(px, py, pz), (int32_t)gpos.size() / 3).first;
                        gpos.push_back(px); gpos.push_back(py); gpos.push_back(pz);
                    }
                    id = nb + it->second;
                }
            }
            nbr[(size_t)b * Q + k] = id;
        }
        if (nbr[(size_t)b * Q + 13] != b)
            return fail(c, LB_EINVAL, "level %d: neighbour table centre entry of block %d is not itself", L.id, b + 1);
        borg[(size_t)b * 3 + 0] = (d->map_x[b] - 1) * 8;
        borg[(size_t)b * 3 + 1] = (d->map_y[b] - 1) * 8;
        borg[(size_t)b * 3 + 2] = (d->map_z[b] - 1) * 8;
    }
    const int32_t ngh = (int32_t)(gpos.size() / 3);
    // The ghost fill's tables (GhostChunk, lb_kernels.h).  Ghost cell s serves
    // direction k when s + c_k lies in a block of the level; which cells of a
    // ghost block serve what follows from which of its 26 neighbours are real.
    struct Served {
        int m;                                             // group
        uint32_t cells;                                    // its cells that serve any direction
        std::vector<std::pair<int, uint32_t>> directions;  // direction, its cells that serve it
        int64_t entries;                                   // number of those cells
    };
    std::unordered_map<uint32_t, std::vector<Served>> patterns;
    auto pattern = [&patterns](uint32_t has_real) -> const std::vector<Served>& {
        auto it = patterns.find(has_real);
        if (it != patterns.end()) return it->second;
        std::vector<Served> out;
        for (int m = 0; m < 64; m++) {
            Served v{m, 0u, {}, 0};
            for (int k = 0; k < Q; k++) {
                uint32_t cells = 0;
                for (int d2 = 0; d2 < 8; d2++) {
                    const int lx = 2 * (m & 3) + (d2 & 1), ly = 2 * ((m >> 2) & 3) + ((d2 >> 1) & 1),
                              lz = 2 * (m >> 4) + (d2 >> 2);
                    const int nx = lx + k % 3 - 1, ny = ly + (k / 3) % 3 - 1, nz = lz + k / 9 - 1;
                    const int ox = nx < 0 ? -1 : (nx > 7 ? 1 : 0), oy = ny < 0 ? -1 : (ny > 7 ? 1 : 0),
                              oz = nz < 0 ? -1 : (nz > 7 ? 1 : 0);
                    if (ox == 0 && oy == 0 && oz == 0) continue;
                    if (has_real & (1u << ((ox + 1) + 3 * (oy + 1) + 9 * (oz + 1)))) cells |= 1u << d2;
                }
                if (cells) v.directions.emplace_back(k, cells);
                v.cells |= cells;
            }
            v.entries = __builtin_popcount(v.cells);
            if (v.cells) out.push_back(std::move(v));
        }
        return patterns.emplace(has_real, std::move(out)).first->second;
    };
    std::vector<int32_t> gpb((size_t)ngh * 8, -1);
    std::vector<uint32_t> ggroup, gpair;
    std::vector<lbk::GhostChunk> gchunk;
    lbk::GhostChunk ch{0, 0, 0, 0, 0};
    int64_t n_entries = 0;
    auto close_chunk = [&]() {
        // a wave's work-items should read one direction of neighbouring groups
        std::sort(gpair.begin() + ch.pair, gpair.end(), [](uint32_t u, uint32_t v) {
            const uint32_t ku = (u >> 6) & 31u, kv = (v >> 6) & 31u;
            return ku != kv ? ku < kv : (u & 63u) < (v & 63u);
        });
        if (ch.n_pairs > 0) gchunk.push_back(ch);
    };
    for (int32_t g = 0; g < ngh; g++) {
        const int64_t px = gpos[(size_t)g * 3], py = gpos[(size_t)g * 3 + 1], pz = gpos[(size_t)g * 3 + 2];
        const int32_t origin[3] = {(int32_t)((px - 1) * 8), (int32_t)((py - 1) * 8), (int32_t)((pz - 1) * 8)};
        borg.insert(borg.end(), origin, origin + 3);
        // parent blocks that hold the 5^3 parent cells origin / 2 + 0..4 (1-based) of its corners
        const Level& P = c->levels[(size_t)L.id - 2];
        for (int s = 0; s < 8; s++) {
            int b3[3];
            bool in = true;
            for (int ax = 0; ax < 3; ax++) {
                b3[ax] = ((origin[ax] / 2 - 1) >> 3) + ((s >> ax) & 1);
                in = in && b3[ax] >= 0 && b3[ax] < P.pd[ax];
            }
            if (!in) continue;
            const int32_t pb =
                P.grid_host[(size_t)b3[0] + (size_t)P.pd[0] * ((size_t)b3[1] + (size_t)P.pd[1] * (size_t)b3[2])];
            if (pb >= (1 << 22)) return fail(c, LB_EINVAL, "level %d: parent block index %d too large", L.id, pb);
            gpb[(size_t)g * 8 + (size_t)s] = pb;
        }
        uint32_t has_real = 0;  // bit (ox+1) + 3(oy+1) + 9(oz+1): that neighbour block is real
        for (int n = 0; n < Q; n++)
            if (n != 13 && real.count(key(px + n % 3 - 1, py + (n / 3) % 3 - 1, pz + n / 9 - 1)))
                has_real |= 1u << n;
        for (const Served& v : pattern(has_real)) {
            if (ch.n_groups == lbk::GHOST_GROUPS || ch.n_pairs + (int)v.directions.size() > lbk::GHOST_PAIRS ||
                g - ch.ghost >= lbk::GHOST_BLOCKS) {
                close_chunk();
                ch = {g, (int32_t)ggroup.size(), (int32_t)gpair.size(), 0, 0};
            }
            const uint32_t gl = (uint32_t)(g - ch.ghost);
            for (const auto& dir : v.directions)
                gpair.push_back((uint32_t)ch.n_groups | (uint32_t)dir.first << 6 | dir.second << 11 | gl << 19);
            uint32_t word = gl | (uint32_t)v.m << 5 | v.cells << 11;
            for (int ax = 0; ax < 3; ax++)
                word |= (uint32_t)((origin[ax] / 8) & 1) << (19 + ax) | (uint32_t)(origin[ax] == 0) << (22 + ax);
            ggroup.push_back(word);
            ch.n_groups++;
            ch.n_pairs = (int16_t)(ch.n_pairs + (int)v.directions.size());
            n_entries += v.entries;
        }
    }
    close_chunk();
    L.ngh = ngh;
    L.n_gchunks = (int32_t)gchunk.size();
    const size_t n4 = (size_t)nb * NC, n5 = ((size_t)nb + ngh) * NC * Q;
    L.wide = c->cfg.wide_offsets != 0 || (n5 + 512) * pop_bytes(c->cfg.storage) >= ((size_t)1 << 32);
    L.wide_g = L.wide;  // thermal populations use the same storage
    for (int i = 0; i < 2; i++) {
        // 512 slots of padding: pulls from a missing neighbour block read a
        // harmless slot up to 200 past the cell's own block
        uint8_t* fb = nullptr;
        RC(dalloc(c, &fb, (n5 + 512) * pop_bytes(c->cfg.storage)));
        L.f[i] = fb;
        RC(dalloc(c, &L.rho[i], n4));
        RC(dalloc(c, &L.vel[i], n4 * 3));
        if (c->cfg.ddf_enabled) {
            uint8_t* gb = nullptr;
            RC(dalloc(c, &gb, (n5 + 512) * pop_bytes(c->cfg.storage)));
            L.g[i] = gb;
            RC(dalloc(c, &L.T[i], n4));
        }
    }
    RC(dalloc(c, &L.obst, n4));
    RC(dalloc(c, &L.sponge, n4));
    if (d->wall_dist) RC(dalloc(c, &L.wall_dist, n4));
    count_as(c, c->bytes, std::max(nb, 1));  // a flag byte per block (they are in the work entries)
    RC(dalloc(c, &L.nbr, (size_t)nb * Q));
    RC(dalloc(c, &L.borg, borg.size()));
    RC(dalloc(c, &L.inv, (size_t)nb));
    const int64_t before_ghosts = c->bytes;
    if (!gchunk.empty()) {
        RC(dalloc(c, &L.gpb, gpb.size()));
        RC(dalloc(c, &L.ggroup, ggroup.size()));
        RC(dalloc(c, &L.gpair, gpair.size()));
        RC(dalloc(c, &L.gchunk, gchunk.size()));
        RC(h2d(c, L.gpb, gpb.data(), gpb.size()));
        RC(h2d(c, L.ggroup, ggroup.data(), ggroup.size()));
        RC(h2d(c, L.gpair, gpair.data(), gpair.size()));
        RC(h2d(c, L.gchunk, gchunk.data(), gchunk.size()));
    }
    RC(ghost_list(c, L.id - 1, L));
    // the ghost fill's tables count per served cell and per ghost block, at
    // least one element each
    {
        const int64_t e = n_entries, gh = n_entries > 0 ? ngh : 0;
        const auto one = [](int64_t n) { return std::max<int64_t>(n, 1); };
        const bool fp32 = c->cfg.storage == LB_STORAGE_FP32;
        const int64_t work = (int64_t)sizeof(lbk::Work) * (fp32 ? (e + 255) / 256 : gh);
        count_as(c, before_ghosts,
                 4 * one(2 * e) + work +
                     (fp32 ? 4 * one(8 * e) : 4 + 4 * (gh + 1) + 4 * one(125 * gh) + 4 * one(gh)));
    }
    const size_t ng = (size_t)d->ptr_dim_x * d->ptr_dim_y * d->ptr_dim_z;
    RC(dalloc(c, &L.grid, ng));
    L.pd[0] = d->ptr_dim_x;
    L.pd[1] = d->ptr_dim_y;
    L.pd[2] = d->ptr_dim_z;
    if (nb > 0) {
        RC(h2d(c, L.nbr, nbr.data(), nbr.size()));
        RC(h2d(c, L.borg, borg.data(), borg.size()));
        // processing order: the storage order, interior blocks (all 26
        // neighbours present, ghosts included) first, then the boundary blocks
        std::vector<int32_t> order;
        order.reserve((size_t)nb);
        for (int pass = 0; pass < 2; pass++)
            for (int32_t b = 0; b < nb; b++) {
                bool interior = true;
                for (int k = 0; k < Q; k++) interior = interior && nbr[(size_t)b * Q + k] >= 0;
                if (interior == (pass == 0)) order.push_back(b);
            }
        L.n_int = 0;
        for (int32_t b : order) {
            bool interior = true;
            for (int k = 0; k < Q; k++) interior = interior && nbr[(size_t)b * Q + k] >= 0;
            if (!interior) break;
            L.n_int++;
        }
        RC(h2d(c, L.inv, inv.data(), inv.size()));
        L.order_host = order;
        L.wflags.assign((size_t)nb, 0);
        for (int32_t i = 0; i < nb; i++) {
            const int32_t blk = order[(size_t)i];
            int32_t f = i < L.n_int ? 0 : lbk::WORK_BOUNDARY;
            for (size_t k = (size_t)blk * NC; k < (size_t)(blk + 1) * NC; k++) {
                if (d->sponge[k] > 0.0f) f |= lbk::WORK_SPONGE;
                if (d->wall_dist && d->wall_dist[k] > 0.0f && d->wall_dist[k] < 10.0f) f |= lbk::WORK_WALL;
                if (d->obstacle[k]) f |= lbk::WORK_SOLID;
            }
            L.wflags[(size_t)blk] = f;
        }
        std::vector<lbk::Work> wcol((size_t)nb);
        for (int32_t i = 0; i < nb; i++)
            wcol[(size_t)i] = mkwork(L.id - 1, order[(size_t)i], 0, L.nbr + (size_t)order[(size_t)i] * Q,
                                     L.wflags[(size_t)order[(size_t)i]]);
        RC(dalloc(c, &L.wcol, wcol.size()));
        RC(h2d(c, L.wcol, wcol.data(), wcol.size()));
        RC(h2d(c, L.obst, d->obstacle, n4));
        RC(h2d(c, L.sponge, d->sponge, n4));
        if (d->wall_dist) RC(h2d(c, L.wall_dist, d->wall_dist, n4));
    }
    if (ng > 0) {
        std::vector<int32_t> grid(ng);
        for (size_t i = 0; i < ng; i++) {
            int v = d->block_pointer[i];
            if (v < 0 || v > nb) return fail(c, LB_EINVAL, "level %d: block_pointer entry out of range", L.id);
            grid[i] = v - 1;
        }
        RC(h2d(c, L.grid, grid.data(), ng));
        L.grid_host = std::move(grid);
    }
    const int64_t before_links = c->bytes;
    RC(build_links(c, L, d));
    RC(link_list(c, L.id - 1, L));
    // the links count 3 slots, 2 weights and 1 value each, and a work entry per 256
    count_as(c, before_links,
             L.nlinks * (3 * (L.lidx32 ? 4 : 8) + 12) + (L.nlinks + 255) / 256 * (int64_t)sizeof(lbk::Work));
    RC(upload_level_args(c, L.id - 1));
    L.uploaded = true;
    return LB_OK;
}

int lb_init_equilibrium(lb_ctx* c, float T0) {
    lbsync::SetupGuard guard;
    RC(check_ctx(c));
    HIPCHK(c, hipSetDevice(c->device));
    for (auto& L : c->levels) {
        HIPCHK(c, c->k->init_level(L.f[0], L.f[1], L.rho[0], L.rho[1], L.vel[0], L.vel[1], L.nb, c->cfg.storage,
                                   c->stream));
        if (c->cfg.ddf_enabled)
            HIPCHK(c, c->k->init_thermal(L.g[0], L.g[1], L.T[0], L.T[1], L.nb, T0, c->cfg.storage, c->stream));
        L.cur = 0;
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return LB_OK;
}

int lb_step_batch(lb_ctx* c, int64_t t_start, int32_t n_steps, float u_curr, const lb_step_params* p) {
    lbsync::SetupGuard guard;
    RC(check_ctx(c));
    if (!p || n_steps < 0 || t_start < 0) return fail(c, LB_EINVAL, "bad step arguments");
    HIPCHK(c, hipSetDevice(c->device));
    // One record for the whole call: coarse step t_start + i starts at substep
    // i of level 1.  A record per coarse step was a launch of 5 us each (of 42
    // us for 55 k cells, 330 us for 1.3 M).
    if (n_steps > 0) queued_steps(&c->queued);
    if (n_steps > 0) HIPCHK(c, c->k->set_state(c->st_dev, case_record(t_start, u_curr, p, c->cfg), c->stream));
    for (int32_t i = 0; i < n_steps; i++) {
        RC(step_level(c, 0, i));
        set_current(c, t_start + i);
    }
    return LB_OK;
}

int lb_synchronize(lb_ctx* c) {
    lbsync::SetupGuard guard;
    if (!c) return LB_EINVAL;
    HIPCHK(c, hipSetDevice(c->device));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return LB_OK;
}

int lb_mesh_upload(lb_ctx* c, int64_t n, const float* cx, const float* cy, const float* cz, const float* nx,
                   const float* ny, const float* nz, const float* areas) {
    lbsync::SetupGuard guard;
    if (!c || n < 0 || (!c->dry && n > 0 && (!cx || !cy || !cz || !nx || !ny || !nz || !areas))) return LB_EINVAL;
    if (c->n_tri != 0) return fail(c, LB_ESTATE, "mesh already uploaded");
    if (!c->dry) HIPCHK(c, hipSetDevice(c->device));
    const float* src[7] = {cx, cy, cz, nx, ny, nz, areas};
    for (int i = 0; i < 7; i++) {
        RC(dalloc(c, &c->mesh[i], (size_t)n));
        if (n > 0) RC(h2d(c, c->mesh[i], src[i], (size_t)n));
    }
    for (int i = 0; i < 4; i++) RC(dalloc(c, &c->maps[i], (size_t)n));
    int groups = (int)((n + 255) / 256);
    RC(dalloc(c, &c->fpart, (size_t)std::max(groups, 1) * 9));
    c->n_tri = n;
    return LB_OK;
}

}  // extern "C"

namespace {
// The force kernel's arguments on the finest level for one side of the surface.
lbk::ForceArgs force_args(lb_ctx* c, const lb_force_params* fp, float side) {
    const Level& L = c->levels.back();
    lbk::ForceArgs a;
    std::memset(&a, 0, sizeof a);
    a.rho = L.rho[L.cur];
    a.vel = L.vel[0];  // level.vel, as surface.jl:784 reads it
    a.obst = L.obst;
    a.grid = L.grid;
    a.gdx = L.pd[0];
    a.gdy = L.pd[1];
    a.gdz = L.pd[2];
    a.dx = (float)L.dx;
    a.n_tri = c->n_tri;
    a.cx = c->mesh[0]; a.cy = c->mesh[1]; a.cz = c->mesh[2];
    a.nx = c->mesh[3]; a.ny = c->mesh[4]; a.nz = c->mesh[5];
    a.area = c->mesh[6];
    a.off_x = (float)fp->mesh_offset[0];
    a.off_y = (float)fp->mesh_offset[1];
    a.off_z = (float)fp->mesh_offset[2];
    const float ps = (float)(fp->rho_physical * fp->velocity_scale * fp->velocity_scale);
    a.pressure_scale = ps;
    a.stress_scale = ps;
    a.tau_mol = L.tau;
    a.search_radius = fp->search_radius;
    a.c_wale = fp->c_wale;
    a.nu_sgs_bg = fp->nu_sgs_background;
    a.ref_x = (float)fp->moment_center[0];
    a.ref_y = (float)fp->moment_center[1];
    a.ref_z = (float)fp->moment_center[2];
    a.p_map = c->maps[0];
    a.sx_map = c->maps[1];
    a.sy_map = c->maps[2];
    a.sz_map = c->maps[3];
    a.partials = c->fpart;
    a.side = side;
    return a;
}
}  // namespace

extern "C" {

int lb_forces(lb_ctx* c, const lb_force_params* fp, double* out, float* p_map, float* sx_map, float* sy_map,
              float* sz_map) {
    lbsync::SetupGuard guard;
    RC(check_ctx(c));
    if (!fp || !out) return fail(c, LB_EINVAL, "null argument");
    if (c->n_tri <= 0) return fail(c, LB_ESTATE, "no mesh uploaded");
    HIPCHK(c, hipSetDevice(c->device));
    const lbk::ForceArgs a = force_args(c, fp, 1.0f);
    const int groups = (int)((c->n_tri + 255) / 256);
    HIPCHK(c, c->k->forces(a, groups, nullptr, c->stream));
    std::vector<double> part((size_t)groups * 9);
    HIPCHK(c, hipMemcpyAsync(part.data(), c->fpart, part.size() * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    if (p_map) HIPCHK(c, hipMemcpyAsync(p_map, c->maps[0], (size_t)c->n_tri * 4, hipMemcpyDeviceToHost, c->stream));
    if (sx_map) HIPCHK(c, hipMemcpyAsync(sx_map, c->maps[1], (size_t)c->n_tri * 4, hipMemcpyDeviceToHost, c->stream));
    if (sy_map) HIPCHK(c, hipMemcpyAsync(sy_map, c->maps[2], (size_t)c->n_tri * 4, hipMemcpyDeviceToHost, c->stream));
    if (sz_map) HIPCHK(c, hipMemcpyAsync(sz_map, c->maps[3], (size_t)c->n_tri * 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    double s[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int g = 0; g < groups; g++)
        for (int j = 0; j < 9; j++) s[j] += part[(size_t)g * 9 + j];
    double Fxp = s[0], Fyp = s[1], Fzp = s[2], Fxv = s[3], Fyv = s[4], Fzv = s[5], Mx = s[6], My = s[7], Mz = s[8];
    // integrate_surface_forces! (surface.jl:873-910)
    if (fp->symmetric) {
        Fxp *= 2.0; Fzp *= 2.0; Fxv *= 2.0; Fzv *= 2.0; My *= 2.0;
        Fyp = 0.0; Fyv = 0.0; Mx = 0.0; Mz = 0.0;
    }
    out[LB_F_FXP] = Fxp; out[LB_F_FYP] = Fyp; out[LB_F_FZP] = Fzp;
    out[LB_F_FXV] = Fxv; out[LB_F_FYV] = Fyv; out[LB_F_FZV] = Fzv;
    out[LB_F_MX] = Mx; out[LB_F_MY] = My; out[LB_F_MZ] = Mz;
    out[LB_F_FX] = Fxp + Fxv; out[LB_F_FY] = Fyp + Fyv; out[LB_F_FZ] = Fzp + Fzv;
    double q_inf = 0.5 * fp->rho_ref * fp->u_ref * fp->u_ref;
    double F_ref = q_inf * fp->area_ref;
    double M_ref = F_ref * fp->chord_ref;
    out[LB_F_CD] = out[LB_F_CL] = out[LB_F_CS] = 0.0;
    out[LB_F_CMX] = out[LB_F_CMY] = out[LB_F_CMZ] = 0.0;
    if (F_ref > 1e-10) {
        out[LB_F_CD] = out[LB_F_FX] / F_ref;
        out[LB_F_CL] = out[LB_F_FZ] / F_ref;
        out[LB_F_CS] = out[LB_F_FY] / F_ref;
    }
    if (M_ref > 1e-10) {
        out[LB_F_CMX] = Mx / M_ref;
        out[LB_F_CMY] = My / M_ref;
        out[LB_F_CMZ] = Mz / M_ref;
    }
    return LB_OK;
}

int lb_surface_maps(lb_ctx* c, const lb_force_params* fp, int32_t side, float* p_map, float* sx_map, float* sy_map,
                    float* sz_map) {
    lbsync::SetupGuard guard;
    RC(check_ctx(c));
    if (!fp || !p_map || !sx_map || !sy_map || !sz_map) return fail(c, LB_EINVAL, "null argument");
    if (side != 1 && side != -1) return fail(c, LB_EINVAL, "side must be +1 or -1");
    if (c->n_tri <= 0) return fail(c, LB_ESTATE, "no mesh uploaded");
    HIPCHK(c, hipSetDevice(c->device));
    const lbk::ForceArgs a = force_args(c, fp, (float)side);
    const int groups = (int)((c->n_tri + 255) / 256);
    HIPCHK(c, c->k->forces(a, groups, nullptr, c->stream));
    float* dst[4] = {p_map, sx_map, sy_map, sz_map};
    for (int m = 0; m < 4; m++)
        HIPCHK(c, hipMemcpyAsync(dst[m], c->maps[m], (size_t)c->n_tri * 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return LB_OK;
}

int lb_download_level(lb_ctx* c, int level_id, int field, float* dst) {
    lbsync::SetupGuard guard;
    RC(check_ctx(c));
    if (!dst || level_id < 1 || level_id > (int)c->levels.size()) return fail(c, LB_EINVAL, "bad arguments");
    HIPCHK(c, hipSetDevice(c->device));
    const Level& L = c->levels[(size_t)level_id - 1];
    HIPCHK(c, hipStreamSynchronize(c->stream));
    const void* src = nullptr;
    int n_comp = 1, storage = LB_STORAGE_FP32;
    bool population = false;
    switch (field) {
        case LB_FIELD_F:
        case LB_FIELD_G:
            src = field == LB_FIELD_F ? L.f[L.cur] : L.g[L.cur];
            n_comp = Q;
            storage = c->cfg.storage;
            population = true;
            break;
        case LB_FIELD_RHO:
            src = L.rho[L.cur];
            break;
        case LB_FIELD_T:
            src = L.T[L.cur];
            break;
        case LB_FIELD_VEL:
            src = L.vel[L.cur];
            n_comp = 3;
            break;
        default:
            return fail(c, LB_EINVAL, "unknown field %d", field);
    }
    if (!src) return fail(c, LB_EINVAL, "field not allocated");
    return download_field(c, L, src, n_comp, storage, population, dst);
}

// Overwrite the current state of a level (both halves of the ping-pong pair,
// so the next step reads it whatever its parity).
int lb_upload_level(lb_ctx* c, int level_id, int field, const float* src) {
    lbsync::SetupGuard guard;
    RC(check_ctx(c));
    if (!src || level_id < 1 || level_id > (int)c->levels.size()) return fail(c, LB_EINVAL, "bad arguments");
    HIPCHK(c, hipSetDevice(c->device));
    Level& L = c->levels[(size_t)level_id - 1];
    const size_t n4 = (size_t)L.nb * NC;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    std::vector<float> tmp;
    float* const* pair;
    size_t n;
    switch (field) {
        case LB_FIELD_F:
        case LB_FIELD_G: {
            void* const dev[2] = {field == LB_FIELD_F ? L.f[0] : L.g[0], field == LB_FIELD_F ? L.f[1] : L.g[1]};
            if (!dev[0]) return fail(c, LB_EINVAL, "field not allocated");
            const int st = c->cfg.storage;
            std::vector<uint8_t> raw(n4 * Q * pop_bytes(st));
            for (int k = 0; k < Q; k++) {
                const float w = wk_host(k);
                for (int64_t b = 0; b < L.nb; b++) {
                    const float* in = src + (size_t)k * n4 + (size_t)L.perm[(size_t)b] * NC;
                    for (int cl = 0; cl < NC; cl++) encode_pop(raw.data(), fidx(b, k, cl), in[cl], st, w);
                }
            }
            for (int i = 0; i < 2; i++) HIPCHK(c, hipMemcpy(dev[i], raw.data(), raw.size(), hipMemcpyHostToDevice));
            return LB_OK;
        }
        case LB_FIELD_RHO:
        case LB_FIELD_T:
            pair = field == LB_FIELD_RHO ? L.rho : L.T;
            if (!pair[0]) return fail(c, LB_EINVAL, "field not allocated");
            tmp.resize(n4);
            for (int64_t b = 0; b < L.nb; b++)
                std::memcpy(tmp.data() + (size_t)b * NC, src + (size_t)L.perm[(size_t)b] * NC, NC * 4);
            n = n4;
            break;
        case LB_FIELD_VEL:
            pair = L.vel;
            tmp.resize(n4 * 3);
            for (int64_t b = 0; b < L.nb; b++)
                for (int d = 0; d < 3; d++)
                    std::memcpy(tmp.data() + ((size_t)b * 3 + d) * NC, src + (size_t)d * n4 + (size_t)L.perm[(size_t)b] * NC,
                                NC * 4);
            n = tmp.size();
            break;
        default:
            return fail(c, LB_EINVAL, "unknown field %d", field);
    }
    for (int i = 0; i < 2; i++) HIPCHK(c, hipMemcpy(pair[i], tmp.data(), n * 4, hipMemcpyHostToDevice));
    return LB_OK;
}

int lb_stats(lb_ctx* c, int level_id, double* out) {
    lbsync::SetupGuard guard;
    RC(check_ctx(c));
    if (!out || level_id < 1 || level_id > (int)c->levels.size()) return fail(c, LB_EINVAL, "bad arguments");
    HIPCHK(c, hipSetDevice(c->device));
    const Level& L = c->levels[(size_t)level_id - 1];
    const int groups = std::max(1, std::min<int>(L.nb, kStatsRows));
    if (c->n_stat_groups < groups) {
        RC(dalloc(c, &c->spart, (size_t)kStatsRows * 8));
        c->n_stat_groups = kStatsRows;
    }
    for (int i = 0; i < 8; i++) out[i] = 0;
    if (L.nb == 0) return LB_OK;
    HIPCHK(c, c->k->stats(L.f[L.cur], L.rho[L.cur], L.vel[L.cur], L.obst, L.nb, c->cfg.storage, c->spart, groups,
                          c->stream));
    std::vector<double> part((size_t)groups * 8);
    HIPCHK(c, hipMemcpyAsync(part.data(), c->spart, part.size() * 8, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    double mn = 1e300, mx = -1e300, vmax = 0;
    for (int g = 0; g < groups; g++) {
        const double* q = &part[(size_t)g * 8];
        out[0] += q[0];
        out[1] += q[1];
        mn = std::min(mn, q[2]);
        mx = std::max(mx, q[3]);
        out[4] += q[4];
        out[5] += q[5];
        out[6] += q[6];
        vmax = std::max(vmax, q[7]);
    }
    out[2] = mn;
    out[3] = mx;
    out[7] = vmax;
    return LB_OK;
}

int lb_check_finite(lb_ctx* c, int64_t* n_nonfinite) {
    lbsync::SetupGuard guard;
    RC(check_ctx(c));
    HIPCHK(c, hipSetDevice(c->device));
    std::vector<lbk::FiniteEntry> ents;
    for (const Level& L : c->levels)
        if (L.nb > 0) ents.push_back(finite_entry(L, L.cur, 0));
    int32_t count = 0;
    if (!ents.empty()) {
        HIPCHK(c, hipMemcpyAsync(c->fin_ents, ents.data(), ents.size() * sizeof(lbk::FiniteEntry),
                                 hipMemcpyHostToDevice, c->stream));
        HIPCHK(c, hipMemsetAsync(c->fin_count, 0, sizeof(int32_t), c->stream));
        HIPCHK(c, c->k->finite_count(c->fin_ents, (int32_t)ents.size(), largest(ents), c->fin_count, c->stream));
        HIPCHK(c, hipMemcpyAsync(&count, c->fin_count, sizeof(int32_t), hipMemcpyDeviceToHost, c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
    }
    if (n_nonfinite) *n_nonfinite = count;
    if (count > 0) return fail(c, LB_ENONFINITE, "%d non-finite density/velocity values", count);
    return LB_OK;
}

int lb_stats_noalloc(lb_ctx* c, int level_id, double* out) {
    lbsync::SetupGuard guard;
    RC(check_ctx(c));
    if (!out || level_id < 1 || level_id > (int)c->levels.size()) return fail(c, LB_EINVAL, "bad arguments");
    HIPCHK(c, hipSetDevice(c->device));
    const Level& L = c->levels[(size_t)level_id - 1];
    const int groups = std::max(1, std::min<int>(L.nb, kStatsRows));
    if (groups > kStatsRows)
        return fail(c, LB_EINVAL, "lb_stats_noalloc: %d partial rows exceed the scratch of %d", groups, kStatsRows);
    for (int i = 0; i < 8; i++) out[i] = 0;
    if (L.nb == 0) return LB_OK;
    hipError_t se = hipSuccess;
    double* s = scratch_on(c->device, &se);
    if (!s) return fail(c, LB_EHIP, "lb_stats_noalloc: no scratch address on device %d (%s)", c->device,
                        hipGetErrorString(se));
    HIPCHK(c, c->k->stats(L.f[L.cur], L.rho[L.cur], L.vel[L.cur], L.obst, L.nb, c->cfg.storage, s, groups,
                          c->stream));
    double* res = s + (size_t)kStatsRows * 8;
    hipLaunchKernelGGL(stats_reduce_kernel, dim3(1), dim3(64), 0, c->stream, s, groups, res);
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipMemcpyAsync(out, res, 8 * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return LB_OK;
}

int64_t lb_device_bytes(const lb_ctx* c) { return c ? c->bytes : 0; }

int lb_profile_enable(lb_ctx* c, int enable) {
    if (!c) return LB_EINVAL;
    c->profile = enable != 0;
    return LB_OK;
}

int lb_profile_read_kernel(lb_ctx* c, int level_id, int kernel, double* ms, int64_t* launches) {
    lbsync::SetupGuard guard;
    if (!c || !ms || !launches || level_id < 1 || level_id > (int)c->levels.size() || kernel < 0 || kernel > 1)
        return LB_EINVAL;
    HIPCHK(c, hipSetDevice(c->device));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    Level& L = c->levels[(size_t)level_id - 1];
    double tot = 0.0;
    for (size_t i = 0; i < L.ev_used[kernel]; i++) {
        float t = 0.0f;
        HIPCHK(c, hipEventElapsedTime(&t, L.ev[kernel][i].first, L.ev[kernel][i].second));
        tot += (double)t;
    }
    *ms = tot;
    *launches = (int64_t)L.ev_used[kernel];
    L.ev_used[kernel] = 0;
    return LB_OK;
}

int lb_profile_read(lb_ctx* c, int level_id, double* ms, int64_t* launches) {
    return lb_profile_read_kernel(c, level_id, 0, ms, launches);
}

int lb_engine_create(lb_engine** out, int device, int32_t storage, int32_t strict_fp) {
    lbsync::SetupGuard guard;
    if (!out) return LB_EINVAL;
    *out = nullptr;
    if (storage < LB_STORAGE_FP32 || storage > LB_STORAGE_BF16) return LB_EINVAL;
    lb_engine* e = new lb_engine();
    e->device = device;
    e->storage = storage;
    e->waves = default_waves(storage);
    e->k = strict_fp ? &kStrict : &kFast;
    if (hipSetDevice(device) != hipSuccess || hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking) != hipSuccess) {
        delete e;
        return LB_EHIP;
    }
    queued_open(&e->queued, e->stream);
    *out = e;
    return LB_OK;
}

void lb_engine_destroy(lb_engine* e) {
    lbsync::SetupGuard guard;
    if (!e) return;
    (void)hipSetDevice(e->device);
    (void)hipStreamSynchronize(e->stream);
    for (EngineCase& ec : e->cases) ec.c->engine = nullptr;
    engine_free_lists(e);
    if (e->fin_ents) (void)hipFree(e->fin_ents);
    if (e->fin_counts) (void)hipFree(e->fin_counts);
    queued_close(&e->queued);
    (void)hipStreamDestroy(e->stream);
    delete e;
}

const char* lb_engine_last_error(const lb_engine* e) { return e ? e->err.c_str() : "null engine"; }

int lb_engine_add(lb_engine* e, lb_ctx* c, int64_t n_coarse_steps, const float* u_batches, int32_t n_batches,
                  int32_t batch_len, const lb_step_params* p) {
    lbsync::SetupGuard guard;
    if (!e || !c || !u_batches || !p) return LB_EINVAL;
    RC(check_ctx(c));
    if (c->device != e->device) return efail(e, LB_EINVAL, "case is on device %d, engine on %d", c->device, e->device);
    if (c->cfg.storage != e->storage) return efail(e, LB_EINVAL, "case storage differs from the engine's");
    if ((c->k == &kStrict) != (e->k == &kStrict)) return efail(e, LB_EINVAL, "case and engine builds differ");
    if (n_coarse_steps < 1 || batch_len < 1 || (int64_t)n_batches * batch_len < n_coarse_steps)
        return efail(e, LB_EINVAL, "bad step count or ramp table");
    EHIPCHK(e, hipSetDevice(e->device));
    EHIPCHK(e, hipStreamSynchronize(c->stream));
    EngineCase ec;
    ec.c = c;
    ec.n_total = n_coarse_steps;
    ec.t0 = 1;
    ec.batch = batch_len;
    ec.p = *p;
    if (dalloc(c, &ec.u_tab, (size_t)n_batches) != LB_OK) return efail(e, LB_ENOMEM, "%s", c->err.c_str());
    if (h2d(c, ec.u_tab, u_batches, (size_t)n_batches) != LB_OK) return efail(e, LB_EHIP, "%s", c->err.c_str());
    if (dalloc(c, &ec.acc, 10) != LB_OK) return efail(e, LB_ENOMEM, "%s", c->err.c_str());
    EHIPCHK(e, hipMemset(ec.acc, 0, 10 * sizeof(double)));
    c->engine = e;
    e->cases.push_back(ec);
    e->dirty = true;
    return LB_OK;
}

int lb_engine_remove(lb_engine* e, lb_ctx* c) {
    lbsync::SetupGuard guard;
    if (!e || !c) return LB_EINVAL;
    EHIPCHK(e, hipSetDevice(e->device));
    for (size_t i = 0; i < e->cases.size(); i++) {
        if (e->cases[i].c != c) continue;
        EHIPCHK(e, hipStreamSynchronize(e->stream));
        const int64_t done = std::min(e->cases[i].t0 - 1, e->cases[i].n_total);
        if (done >= 1) set_current(c, done);
        c->engine = nullptr;
        e->cases.erase(e->cases.begin() + (long)i);
        e->dirty = true;
        return LB_OK;
    }
    return efail(e, LB_EINVAL, "case is not attached to this engine");
}

int lb_engine_step(lb_engine* e, int32_t n) {
    if (!e || n < 0) return LB_EINVAL;
    EHIPCHK(e, hipSetDevice(e->device));
    if (e->cases.empty() || n == 0) return LB_OK;
    if (e->dirty) {
        lbsync::SetupGuard guard;
        RC(engine_rebuild(e));
    }
    queued_steps(&e->queued);
    if (e->use_graph && !e->exec) {
        // GPU calls of other threads wait for the capture (lb_sync.h);
        // relaxed mode in addition lets them run host-side work meanwhile
        std::unique_lock<lbsync::CaptureLock> capture(lbsync::capture_mutex());
        EHIPCHK(e, hipStreamBeginCapture(e->stream, hipStreamCaptureModeRelaxed));
        const hipError_t r = engine_issue_step(e);
        hipGraph_t g = nullptr;
        const hipError_t r2 = hipStreamEndCapture(e->stream, &g);
        if (r != hipSuccess || r2 != hipSuccess) {
            if (g) (void)hipGraphDestroy(g);
            return efail(e, LB_EHIP, "graph capture failed: %s", hipGetErrorString(r != hipSuccess ? r : r2));
        }
        e->graph = g;
        EHIPCHK(e, hipGraphInstantiate(&e->exec, e->graph, nullptr, nullptr, 0));
    }
    for (int32_t i = 0; i < n; i++) {
        if (e->use_graph) EHIPCHK(e, hipGraphLaunch(e->exec, e->stream));
        else EHIPCHK(e, engine_issue_step(e));
        for (EngineCase& ec : e->cases)
            if (ec.t0 <= ec.n_total) ec.t0 += ec.t_inc;
    }
    return LB_OK;
}

int lb_engine_synchronize(lb_engine* e) {
    lbsync::SetupGuard guard;
    if (!e) return LB_EINVAL;
    EHIPCHK(e, hipSetDevice(e->device));
    EHIPCHK(e, hipStreamSynchronize(e->stream));
    return LB_OK;
}

int lb_engine_case_progress(const lb_engine* e, const lb_ctx* c, int64_t* t_done) {
    if (!e || !c || !t_done) return LB_EINVAL;
    for (const EngineCase& ec : e->cases)
        if (ec.c == c) {
            *t_done = std::min(ec.t0 - 1, ec.n_total);
            return LB_OK;
        }
    return LB_EINVAL;
}

int lb_engine_sample_forces(lb_engine* e, lb_ctx* c, const lb_force_params* fp, int64_t diag_freq,
                            int64_t ramp_steps) {
    lbsync::SetupGuard guard;
    if (!e || !c || !fp || diag_freq < 1 || ramp_steps < 0) return LB_EINVAL;
    for (EngineCase& ec : e->cases) {
        if (ec.c != c) continue;
        if (c->n_tri <= 0) return efail(e, LB_ESTATE, "case has no mesh");
        EHIPCHK(e, hipSetDevice(e->device));
        EHIPCHK(e, hipStreamSynchronize(e->stream));
        ec.sample = true;
        ec.diag = diag_freq;
        ec.ramp = ramp_steps;
        ec.fp = *fp;
        e->dirty = true;
        return LB_OK;
    }
    return efail(e, LB_EINVAL, "case is not attached to this engine");
}

int lb_engine_case_forces(lb_engine* e, const lb_ctx* c, double* sums, int64_t* n_samples) {
    lbsync::SetupGuard guard;
    if (!e || !c || !sums || !n_samples) return LB_EINVAL;
    for (const EngineCase& ec : e->cases) {
        if (ec.c != c) continue;
        EHIPCHK(e, hipSetDevice(e->device));
        EHIPCHK(e, hipStreamSynchronize(e->stream));
        double acc[10];
        EHIPCHK(e, hipMemcpy(acc, ec.acc, sizeof acc, hipMemcpyDeviceToHost));
        for (int i = 0; i < 9; i++) sums[i] = acc[i];
        // integrate_surface_forces! (surface.jl:873-910) doubles the half model
        if (ec.fp.symmetric) {
            sums[0] *= 2.0; sums[2] *= 2.0; sums[3] *= 2.0; sums[5] *= 2.0; sums[7] *= 2.0;
            sums[1] = 0.0; sums[4] = 0.0; sums[6] = 0.0; sums[8] = 0.0;
        }
        *n_samples = (int64_t)acc[9];
        return LB_OK;
    }
    return efail(e, LB_EINVAL, "case is not attached to this engine");
}

int lb_engine_check_finite(lb_engine* e, lb_ctx** diverged, int32_t cap, int32_t* n_diverged) {
    lbsync::SetupGuard guard;
    if (!e || !n_diverged || cap < 0 || (cap > 0 && !diverged)) return LB_EINVAL;
    *n_diverged = 0;
    EHIPCHK(e, hipSetDevice(e->device));
    EHIPCHK(e, hipStreamSynchronize(e->stream));
    const size_t nc = e->cases.size();
    if (nc == 0) return LB_OK;
    std::vector<lbk::FiniteEntry> ents;
    for (size_t i = 0; i < nc; i++) {
        const EngineCase& ec = e->cases[i];
        const int64_t done = std::min(ec.t0 - 1, ec.n_total);
        for (size_t li = 0; li < ec.c->levels.size(); li++) {
            const Level& L = ec.c->levels[li];
            if (L.nb == 0) continue;
            // output buffer of the level's last substep in coarse step `done`
            const int64_t last = (done << li) + ((int64_t)1 << li) - 1;
            ents.push_back(finite_entry(L, done >= 1 ? 1 - (int)(last & 1) : L.cur, (int32_t)i));
        }
    }
    if (ents.size() > e->fin_cap_ents || nc > e->fin_cap_cases) {
        if (e->fin_ents) (void)hipFree(e->fin_ents);
        if (e->fin_counts) (void)hipFree(e->fin_counts);
        e->fin_ents = nullptr;
        e->fin_counts = nullptr;
        e->fin_cap_ents = e->fin_cap_cases = 0;
        const size_t ce = std::max<size_t>(ents.size(), 64), cc = std::max<size_t>(nc, 16);
        EHIPCHK(e, hipMalloc((void**)&e->fin_ents, ce * sizeof(lbk::FiniteEntry)));
        EHIPCHK(e, hipMalloc((void**)&e->fin_counts, cc * sizeof(int32_t)));
        e->fin_cap_ents = ce;
        e->fin_cap_cases = cc;
    }
    std::vector<int32_t> counts(nc, 0);
    EHIPCHK(e, hipMemcpyAsync(e->fin_ents, ents.data(), ents.size() * sizeof(lbk::FiniteEntry), hipMemcpyHostToDevice,
                              e->stream));
    EHIPCHK(e, hipMemsetAsync(e->fin_counts, 0, nc * sizeof(int32_t), e->stream));
    EHIPCHK(e, e->k->finite_count(e->fin_ents, (int32_t)ents.size(), largest(ents), e->fin_counts, e->stream));
    EHIPCHK(e, hipMemcpyAsync(counts.data(), e->fin_counts, nc * sizeof(int32_t), hipMemcpyDeviceToHost, e->stream));
    EHIPCHK(e, hipStreamSynchronize(e->stream));
    int32_t n = 0;
    for (size_t i = 0; i < nc; i++)
        if (counts[i] > 0) {
            if (n < cap) diverged[n] = e->cases[i].c;
            n++;
        }
    *n_diverged = n;
    if (n > 0) return efail(e, LB_ENONFINITE, "%d case(s) hold non-finite density/velocity values", n);
    return LB_OK;
}

int lb_engine_set_options(lb_engine* e, int32_t use_graph, int32_t schedule, int32_t waves) {
    if (!e || (schedule != LB_SCHED_XCD && schedule != LB_SCHED_LINEAR && schedule != LB_SCHED_PERSISTENT) ||
        waves < 5 || waves > 6)
        return LB_EINVAL;
    EHIPCHK(e, hipSetDevice(e->device));
    EHIPCHK(e, hipStreamSynchronize(e->stream));
    e->use_graph = use_graph != 0;
    e->sched = schedule;
    e->waves = waves;
    // the captured graph bakes the schedule in
    if (e->exec) (void)hipGraphExecDestroy(e->exec);
    if (e->graph) (void)hipGraphDestroy(e->graph);
    e->exec = nullptr;
    e->graph = nullptr;
    return LB_OK;
}

// Device bytes a case will hold: the allocations of lb_create,
// lb_level_upload (every level) and lb_mesh_upload, counted by running the
// same host code without allocating (no GPU needed), plus the engine's ramp
// table of n_ramp_batches values.  lb_stats adds 65,536 bytes on first use.
int lb_footprint(const lb_config* cfg, const lb_level_desc* levels, int32_t n_levels, int64_t n_tri,
                 int32_t n_ramp_batches, int64_t* bytes) {
    if (!cfg || !levels || !bytes || n_levels != cfg->n_levels || n_levels < 1 || n_levels > 16) return LB_EINVAL;
    lb_ctx c;
    c.dry = true;
    c.cfg = *cfg;
    c.levels.resize((size_t)n_levels);
    c.las_host.resize((size_t)n_levels);
    RC(create_buffers(&c));
    for (int i = 0; i < n_levels; i++) RC(lb_level_upload(&c, &levels[i]));
    if (n_tri > 0) RC(lb_mesh_upload(&c, n_tri, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr));
    if (n_ramp_batches > 0) {
        float* u = nullptr;
        double* acc = nullptr;
        RC(dalloc(&c, &u, (size_t)n_ramp_batches));
        RC(dalloc(&c, &acc, 10));
    }
    *bytes = c.bytes;
    return LB_OK;
}

int lb_device_memory(int device, int64_t* free_bytes, int64_t* total_bytes) {
    lbsync::SetupGuard guard;
    if (!free_bytes || !total_bytes) return LB_EINVAL;
    if (hipSetDevice(device) != hipSuccess) return LB_EHIP;
    size_t f = 0, t = 0;
    if (hipMemGetInfo(&f, &t) != hipSuccess) return LB_EHIP;
    *free_bytes = (int64_t)f;
    *total_bytes = (int64_t)t;
    return LB_OK;
}

}  // extern "C"
