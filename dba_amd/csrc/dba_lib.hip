// dba_lib.hip - C ABI of the MI355X DBA time step (libdba_hip.so).
//
// Host orchestration of the gfx950 kernels: instances own their device state,
// groups merge instances of one model into one worklist, every step is
//   step kernel (fused stencil + detector byte per tile)
//   -> finalize kernel (parity flip, history, conserved shift / CFL dt,
//      compaction of the next worklist),
// on one HIP stream, optionally replayed from a captured hipGraph.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/dba/dba.h"
#include "common.h"
#include "k_finalize.h"
#include "k_ch.h"
#include "k_resident.h"
#include "k_k93.h"
#include "k_resident_k93.h"
#include "k_kh.h"
#include "k_ref3d.h"
#include "k_diag.h"
#include "k_droplets.h"

using namespace dba;

// Device scratch of dba_droplets_noalloc: one array per GPU, held from module
// load until the process ends. Host code reaches it only through the address
// hipGetSymbolAddress returns for the current device (dba_ctx::scratch); the
// name itself is a host-side stand-in, not a device address.
constexpr int64_t kScratchMaxCells = int64_t(1) << 22;  // 2048^2 (161^3) cells
constexpr size_t kScratchTail = 64 * 1024;               // block partials, counters
constexpr size_t kScratchBytes = 13 * (size_t)kScratchMaxCells + kScratchTail;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {

thread_local std::string g_error;

dba_status fail(dba_status code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_error = buf;
    return code;
}

#define HIP_TRY(expr)                                                                  \
    do {                                                                               \
        hipError_t e_ = (expr);                                                        \
        if (e_ != hipSuccess)                                                          \
            return fail(DBA_ERR_HIP, "%s failed: %s", #expr, hipGetErrorString(e_));   \
    } while (0)

#define LAUNCH_CHECK()                                                                 \
    do {                                                                               \
        hipError_t e_ = hipGetLastError();                                             \
        if (e_ != hipSuccess)                                                          \
            return fail(DBA_ERR_LAUNCH, "kernel launch failed: %s", hipGetErrorString(e_)); \
    } while (0)

int nfields_of(int model) {
    switch (model) {
        case DBA_MODEL_CH: return 1;
        case DBA_MODEL_DENDRITE_K93: return 2;
        case DBA_MODEL_KH: return 4;
        case DBA_MODEL_DENDRITE_K94: return 2;
        case DBA_MODEL_MODELB: return 4;
        default: return 0;
    }
}

int nsets_of(int model) {
    return (model == DBA_MODEL_DENDRITE_K93 || model == DBA_MODEL_DENDRITE_K94) ? 2 : 1;
}

bool is_pow2_tile(int t) { return t == 8 || t == 16 || t == 32; }

struct Instance {
    int id = 0;
    dba_params p{};
    Inst h{};                    // host copy of the device descriptor
    void* arena = nullptr;       // the device allocation that holds this instance's arrays
    int64_t footprint = 0;
    int64_t ncell = 0;
    bool needs_prime = false;    // KH: per-tile wave speeds must be recomputed before the next step
    bool stepped = false;        // work for this instance has been enqueued on the compute stream
    Inst* d_self = nullptr;      // single-instance descriptor (downloads, checks)
};

struct Group {
    std::vector<int> ids;
    int model = 0, tile = 0, tile_z = 1, threads = 0;
    int dense_threads = 0;        // workgroup size of the single-launch step kernel
    bool conserved = false;       // one conserved instance (single-launch steps carry its mean shift)
    bool partial = false;         // an instance with partial tiles: the kernels' PART instances
    int march = 0;                // column-march single-launch steps: tiles per strip (0: off)
    bool spec = false;            // K93 single-launch steps with speculative staging
    bool kh_p2 = false;           // KH: dx, dy and the cell area of every instance are powers of two
    int march_from = 0;           // Model B: lists of at least this many blocks take the column march (0: never, 1: the block kernels are not launched)
    int mb_nl = 1, mb_ncx = 0, mb_ncy = 0, mb_ntz = 0;  // ... layers per strip, columns in x and y, layers
    bool nine = true;             // CH 9-point stencil (the march kernel is instanced on it)
    int res_gx = 0, res_gy = 0, res_threads = 0, res_per_tile = 0;  // resident steps (k_resident.h): region, workgroup, threads per tile (0: not taken)
    Inst* d_insts = nullptr;
    Seg* d_segs = nullptr;
    InstSegs* d_isegs = nullptr;
    SegPart* d_parts = nullptr;
    int32_t* d_counts = nullptr;
    int32_t* d_offsets = nullptr;
    int32_t* d_dmap = nullptr;    // single-launch steps of several instances or segments: instance << 24 | tile
    int nseg = 0;
    bool fold = false;            // steps without a merge launch (WorkList::counts)
    int64_t total_tiles = 0;
    int grid = 0;
    uint64_t last_use = 0;
    int32_t* solo_seg = nullptr;  // one instance in one segment: its worklist ...
    uint64_t* solo_rec = nullptr; // ... its neighbour records
    int solo_nt = 0;              // ... and tile count
};

struct GraphKey {
    std::vector<int> ids;
    int chunk;
    int single_launch;  // the mode the graph was captured in
    bool operator<(const GraphKey& o) const {
        if (chunk != o.chunk) return chunk < o.chunk;
        if (single_launch != o.single_launch) return single_launch < o.single_launch;
        return ids < o.ids;
    }
};

}  // namespace

struct CachedGraph {
    hipGraphExec_t exec = nullptr;
    uint64_t last_use = 0;
};

struct dba_ctx {
    int device = 0;
    int n_cu = 256;                // compute units of the device
    hipStream_t stream = nullptr;  // compute stream: steps, finalize, downloads
    hipStream_t setup = nullptr;   // instance and group set-up, uploads of never-stepped instances
    int next_id = 1;
    uint64_t clock = 0;            // LRU clock of the group and graph caches
    std::map<int, Instance*> inst;
    std::map<std::vector<int>, Group*> groups;
    std::map<GraphKey, CachedGraph> graphs;
    double* staging = nullptr;
    size_t staging_n = 0;
    int* d_flag = nullptr;
    double* d_diag = nullptr;      // diagnostics: block partials, results
    int32_t* d_cols = nullptr;     // diagnostics: growth-front columns
    bool timing = false;
    int single_launch = 1;         // single-launch steps: 0 off, 1 one-instance groups, 2 also batches
    std::vector<std::pair<hipEvent_t, hipEvent_t>> ev_step, ev_fin;  // timed intervals (events may be shared)
    std::vector<hipEvent_t> ev_used;  // every event handed out since the timing was last reset
    std::vector<hipEvent_t> ev_pool;
    hipEvent_t markers[8] = {};
    unsigned char* scratch = nullptr;  // this device's address of the scratch array
    // exchange of the resident steps: one workspace for every instance (its launches
    // follow each other on the one stream; sequence numbers never repeat)
    ResHead* xbuf = nullptr;       // the launches' state, then xwords words of frames and flags
    size_t xwords = 0;
    uint32_t xseq = 1;
    int* stuck = nullptr;          // pinned host word: a resident launch was given up
    std::vector<int> unsettled;    // instances with resident launches since the host last waited
    bool resident = true;          // resident steps where they can be had (dba_set_resident)
    int wait_polls = kWaitPolls;   // polls after which one of their waits is given up
    int64_t resident_calls = 0;    // step calls that took them
    int64_t resident_redone = 0;   // steps of launches given up, made again on another path
};

namespace {

// Derived constants: the same C expressions the oracle evaluates.
void derive_constants(const dba_params& p, Inst& h) {
    h.invdx2 = 1.0 / (p.dx * p.dx);
    h.inv6dx2 = 1.0 / (6.0 * p.dx * p.dx);
    h.inv2dx = 1.0 / (2.0 * p.dx);
    h.dt_tau = p.tau != 0.0 ? p.dt / p.tau : 0.0;
    h.alpha_pi = p.alpha / M_PI;
    double jf = (double)p.aniso_j;
    h.cos_jt0 = std::cos(jf * p.theta0);
    h.sin_jt0 = std::sin(jf * p.theta0);
    h.k_epsp = -(p.eps_bar * jf * p.delta);
    if (p.r_x != 0.0 && p.r_y != 0.0 && p.r_z != 0.0) {  // Model B (validated there)
        h.mb_cx = -1.0 + 1.0 / p.r_x;
        h.mb_cy = -1.0 + 1.0 / p.r_y;
        h.mb_cz = -1.0 + 1.0 / p.r_z;
        h.mb_lk = std::log(p.k_eq) / p.r_z;
    }
    h.k94_f0 = 1. / (2 * p.dx);
    h.k94_f1 = 1. / p.dx / p.dx;
    h.k94_f2 = -p.alpha / 3.14159;
    h.k94_f3 = 1. / p.tau;
    h.mb_irx = 1.0 / p.r_x;
    h.mb_iry = 1.0 / p.r_y;
    h.mb_irz = 1.0 / p.r_z;
    h.mb_gel = 0.5 * p.p_gel / (1.0 - p.z_crit);
}

dba_status validate(const dba_params& p) {
    if (nfields_of(p.model) == 0) return fail(DBA_ERR_INVALID, "model %d is not supported", p.model);
    if (p.mode < 0 || p.mode > 2) return fail(DBA_ERR_INVALID, "mode %d invalid", p.mode);
    if (p.nx <= 0 || p.ny <= 0 || p.nz <= 0) return fail(DBA_ERR_INVALID, "grid %dx%dx%d invalid", p.nx, p.ny, p.nz);
    if (p.model == DBA_MODEL_CH || p.model == DBA_MODEL_DENDRITE_K93) {
        if (p.nz != 1) return fail(DBA_ERR_INVALID, "model %d is 2D (nz must be 1)", p.model);
        if (p.tile_x != p.tile_y || !is_pow2_tile(p.tile_x))
            return fail(DBA_ERR_INVALID, "tile must be square 8, 16 or 32 (got %dx%d)", p.tile_x, p.tile_y);
        // a partial last tile needs two cells or more: its neighbours' halos and its
        // own ring stay within the 3x3 tiles around each tile
        if (p.nx % p.tile_x == 1 || p.ny % p.tile_y == 1)
            return fail(DBA_ERR_INVALID, "grid %dx%d leaves a partial tile one cell wide (tile %d)", p.nx, p.ny,
                        p.tile_x);
        if (p.nx < p.tile_x * 1 || p.ny < p.tile_y) return fail(DBA_ERR_INVALID, "grid smaller than a tile");
    }
    if (p.model == DBA_MODEL_KH) {
        if (p.nz != 1) return fail(DBA_ERR_INVALID, "KH is 2D (nz must be 1)");
        if (p.tile_x != p.tile_y || (p.tile_x != 8 && p.tile_x != 16))
            return fail(DBA_ERR_INVALID, "KH tile must be 8x8 or 16x16");
        if (p.nx % p.tile_x || p.ny % p.tile_y)
            return fail(DBA_ERR_INVALID, "grid %dx%d must be a multiple of the tile %d", p.nx, p.ny, p.tile_x);
        if (p.bc_x != DBA_BC_PERIODIC) return fail(DBA_ERR_INVALID, "KH needs periodic x");
        if (p.bc_y != DBA_BC_PERIODIC && p.bc_y != DBA_BC_WALL) return fail(DBA_ERR_INVALID, "KH y: periodic or wall");
        if (p.dt_mode == DBA_DT_CFL && p.mode == DBA_MODE_CONSERVED)
            return fail(DBA_ERR_INVALID, "conserved KH uses a fixed dt");
        if (p.dt_mode == DBA_DT_CFL && !(p.cfl > 0.0)) return fail(DBA_ERR_INVALID, "cfl must be positive");
        if (!(p.gas_gamma > 1.0)) return fail(DBA_ERR_INVALID, "gas_gamma must exceed 1");
        if (p.dy != p.dx) return fail(DBA_ERR_INVALID, "KH needs dy == dx");
    }
    if (p.model == DBA_MODEL_DENDRITE_K94 || p.model == DBA_MODEL_MODELB) {
        const int tz = p.tile_z > 0 ? p.tile_z : 1;
        if (p.tile_x != 4 || p.tile_y != 4 || (tz != 4 && tz != 1) || (tz == 1) != (p.nz == 1))
            return fail(DBA_ERR_INVALID, "reference 3D models use 4x4x4 blocks (4x4x1 when nz == 1)");
        if (p.nx % 4 || p.ny % 4 || p.nz % tz)
            return fail(DBA_ERR_INVALID, "grid %dx%dx%d must be a multiple of the block", p.nx, p.ny, p.nz);
        if (p.bc_x != DBA_BC_PERIODIC || p.bc_y != DBA_BC_PERIODIC || p.bc_z != DBA_BC_PERIODIC)
            return fail(DBA_ERR_INVALID, "reference 3D models are periodic");
        if (p.model == DBA_MODEL_DENDRITE_K94 && p.mode == DBA_MODE_CONSERVED)
            return fail(DBA_ERR_INVALID, "conserved DBA is defined for Model B and KH only");
        if (p.model == DBA_MODEL_MODELB && (p.r_x == 0.0 || p.r_y == 0.0 || p.r_z == 0.0))
            return fail(DBA_ERR_INVALID, "Model B needs nonzero rx, ry, rz");
    }
    if (p.model == DBA_MODEL_CH && p.stencil != 5 && p.stencil != 9)
        return fail(DBA_ERR_INVALID, "CH stencil must be 5 or 9");
    if (p.model == DBA_MODEL_CH && p.mode == DBA_MODE_CONSERVED && p.bc_x != DBA_BC_PERIODIC)
        return fail(DBA_ERR_INVALID, "conserved DBA needs a periodic grid");
    if (p.model == DBA_MODEL_DENDRITE_K93 && (p.aniso_j < 1 || p.aniso_j > 16))
        return fail(DBA_ERR_INVALID, "aniso_j must be in [1,16]");
    if (p.model == DBA_MODEL_DENDRITE_K93 && p.mode == DBA_MODE_CONSERVED)
        return fail(DBA_ERR_INVALID, "conserved DBA is defined for Model B and KH only");
    const bool wide = p.threads == 512 || p.threads == 1024;
    if (p.threads != 0 && p.threads != 64 && p.threads != 128 && p.threads != 256 && !wide)
        return fail(DBA_ERR_INVALID, "threads must be 0, 64, 128, 256, 512 or 1024");
    if (wide && p.model != DBA_MODEL_CH && p.model != DBA_MODEL_DENDRITE_K93)
        return fail(DBA_ERR_INVALID, "512 and 1024 threads are for the CH and Kobayashi-93 models");
    if (p.dx <= 0.0 || p.dt <= 0.0) return fail(DBA_ERR_INVALID, "dx and dt must be positive");
    return DBA_OK;
}

struct Layout {
    int ntx, nty, ntz, nt, nwords;
    int64_t n;
    int nf, nsets, naux;
    int64_t aux_len;  // doubles per aux array
};

Layout layout_of(const dba_params& p) {
    Layout L{};
    int tz = p.tile_z > 0 ? p.tile_z : 1;
    L.ntx = (p.nx + p.tile_x - 1) / p.tile_x;
    L.nty = (p.ny + p.tile_y - 1) / p.tile_y;
    L.ntz = (p.nz + tz - 1) / tz;
    L.nt = L.ntx * L.nty * L.ntz;
    L.nwords = (L.nt + 63) / 64;
    L.n = (int64_t)p.nx * p.ny * p.nz;
    L.nf = nfields_of(p.model);
    L.nsets = nsets_of(p.model);
    L.naux = 0;
    L.aux_len = L.n;
    if (p.model == DBA_MODEL_MODELB) L.naux = 3;  // chemical potentials (every cell, every mode)
    if (p.mode != DBA_MODE_REGULAR) {
        if (p.model == DBA_MODEL_CH) {             // mu ring: one record per tile
            L.naux = 1;
            L.aux_len = (int64_t)L.nt * (4 * p.tile_x - 4);
        }
        if (p.model == DBA_MODEL_KH) {             // edge state of sleeping tiles: one record per tile
            L.naux = 1;
            L.aux_len = (int64_t)L.nt * (p.tile_x == 8 ? KhEdge<8>::R : KhEdge<16>::R);
        }
    }
    return L;
}

int64_t footprint_of(const dba_params& p) {
    Layout L = layout_of(p);
    int64_t b = 0;
    b += 2 * (int64_t)L.nf * L.n * 8;        // double-buffered fields
    b += (int64_t)L.naux * L.aux_len * 8;    // stored neighbour state
    b += 4 * (int64_t)L.nwords * 8 + 2 * (int64_t)L.nt;  // bitmaps + detector bytes
    b += (int64_t)kMaxFields * L.nt * 8;     // tpart
    b += 2 * (int64_t)L.nt * 8;              // tspeed
    b += (int64_t)kMaxFields * 2 * L.nt * 8; // s_tile
    b += 16 * 8 + 4 * 8;                     // scal + ctr
    b += (int64_t)2 * std::max(0, p.history_cap) * 4;
    b += (int64_t)L.nt * 4;                  // seg
    b += (int64_t)L.nt * 8;                  // nbrec
    b += sizeof(Inst);
    return b;
}

// The arrays of an instance, cut from one device allocation: with one each (about 25),
// creating and destroying 16 dendrites of 324^2 to 903^2 cells took 15 of the 57 ms of
// their 1500-step sweep.
struct Arena {
    std::vector<std::pair<void*, size_t>> want;  // where the pointer goes, the array's offset
    size_t bytes = 0;

    template <typename T>
    void add(T** out, size_t count) {
        // (256 bytes: no two arrays share a cache line, and every load width is aligned)
        bytes = (bytes + 255) & ~(size_t)255;
        want.emplace_back((void*)out, bytes);
        bytes += std::max<size_t>(count * sizeof(T), 8);
    }
};

// Allocates and clears the arena and sets its pointers.
dba_status alloc_arena(Instance* in, const Arena& a, hipStream_t setup) {
    void* ptr = nullptr;
    hipError_t e = hipMalloc(&ptr, a.bytes);
    if (e != hipSuccess) return fail(DBA_ERR_NOMEM, "hipMalloc(%zu) failed: %s", a.bytes, hipGetErrorString(e));
    in->arena = ptr;
    e = hipMemsetAsync(ptr, 0, a.bytes, setup);
    if (e != hipSuccess) return fail(DBA_ERR_HIP, "hipMemset failed: %s", hipGetErrorString(e));
    for (const auto& w : a.want) {
        void* at = (unsigned char*)ptr + w.second;
        memcpy(w.first, &at, sizeof(at));
    }
    return DBA_OK;
}

void free_instance(Instance* in) {
    (void)hipFree(in->arena);
    in->arena = nullptr;
}

void free_group(Group* g) {
    (void)hipFree(g->d_insts);
    (void)hipFree(g->d_segs);
    (void)hipFree(g->d_isegs);
    (void)hipFree(g->d_parts);
    (void)hipFree(g->d_counts);
    (void)hipFree(g->d_offsets);
    (void)hipFree(g->d_dmap);
    delete g;
}

bool subset(const std::vector<int>& a, const std::vector<int>& b) {  // every id of a is in b
    for (int x : a)
        if (std::find(b.begin(), b.end(), x) == b.end()) return false;
    return true;
}

// Drops every captured graph that may launch group g (its ids are a subset of
// the graph's instance set).
void drop_graphs_using(dba_ctx* ctx, const std::vector<int>& gids) {
    for (auto it = ctx->graphs.begin(); it != ctx->graphs.end();) {
        if (subset(gids, it->first.ids)) {
            (void)hipGraphExecDestroy(it->second.exec);
            it = ctx->graphs.erase(it);
        } else {
            ++it;
        }
    }
}

void invalidate_groups(dba_ctx* ctx, int id) {
    for (auto it = ctx->groups.begin(); it != ctx->groups.end();) {
        if (std::find(it->first.begin(), it->first.end(), id) != it->first.end()) {
            free_group(it->second);
            it = ctx->groups.erase(it);
        } else {
            ++it;
        }
    }
    drop_graphs_using(ctx, {id});
}

// Bounded caches: a serving loop steps a changing set of instances, and every
// distinct set has its own groups and graphs. Entries not used by the current
// call (last_use < clock) are evicted least recently used first.
constexpr size_t kMaxGroups = 64;
constexpr size_t kMaxGraphs = 32;

void evict_groups(dba_ctx* ctx) {
    while (ctx->groups.size() >= kMaxGroups) {
        auto victim = ctx->groups.end();
        for (auto it = ctx->groups.begin(); it != ctx->groups.end(); ++it)
            if (it->second->last_use < ctx->clock &&
                (victim == ctx->groups.end() || it->second->last_use < victim->second->last_use))
                victim = it;
        if (victim == ctx->groups.end()) return;
        (void)hipStreamSynchronize(ctx->stream);
        drop_graphs_using(ctx, victim->first);
        free_group(victim->second);
        ctx->groups.erase(victim);
    }
}

void evict_graphs(dba_ctx* ctx) {
    while (ctx->graphs.size() >= kMaxGraphs) {
        auto victim = ctx->graphs.end();
        for (auto it = ctx->graphs.begin(); it != ctx->graphs.end(); ++it)
            if (it->second.last_use < ctx->clock &&
                (victim == ctx->graphs.end() || it->second.last_use < victim->second.last_use))
                victim = it;
        if (victim == ctx->graphs.end()) return;
        (void)hipStreamSynchronize(ctx->stream);
        (void)hipGraphExecDestroy(victim->second.exec);
        ctx->graphs.erase(victim);
    }
}

// Workgroup size per (model, tile) measured best on MI355X (CH and Kobayashi-93
// grids of 1024^2 to 4096^2); the workgroup size never changes results.
int default_threads(int model, int tile) {
    if (tile <= 8) return 64;
    if (tile == 16) return (model == DBA_MODEL_CH || model == DBA_MODEL_DENDRITE_K93) ? 128 : 256;
    return model == DBA_MODEL_DENDRITE_K93 ? 512 : 256;
}

// Single-launch steps of K93 16x16 tiles: every tile takes a workgroup, so a
// small grid gains from more threads per tile (a shorter FP64 chain per tile)
// and a large, mostly sleeping one from narrower workgroups (more of them per
// CU). Measured on MI355X: 512^2 (1024 tiles) 512 threads 8.0 us vs 128 threads
// 10.0 us; 1024^2 256 threads 9.9 vs 11.8 us; 2048^2 128 threads best.
int default_dense_threads(int model, int tile, int64_t tiles) {
    if (model == DBA_MODEL_DENDRITE_K93 && tile == 16) return tiles <= 1024 ? 512 : (tiles <= 4096 ? 256 : 128);
    return default_threads(model, tile);
}

// KH: wave speeds of every tile from the current state, and the first CFL dt.
dba_status kh_prime(dba_ctx* ctx, Instance* in) {
    if (in->p.tile_x == 8)
        hipLaunchKernelGGL((kh_prime_kernel<8>), dim3(std::min(in->h.nt, 4096)), dim3(256), 0, ctx->stream,
                           in->d_self, 0);
    else
        hipLaunchKernelGGL((kh_prime_kernel<16>), dim3(std::min(in->h.nt, 4096)), dim3(256), 0, ctx->stream,
                           in->d_self, 0);
    LAUNCH_CHECK();
    hipLaunchKernelGGL(kh_dt_kernel, dim3(1), dim3(256), 0, ctx->stream, in->d_self, 0);
    LAUNCH_CHECK();
    in->needs_prime = false;
    return DBA_OK;
}

void resident_choose(const dba_ctx* ctx, Group* g, const Inst& h);  // below, with the launches

dba_status get_group(dba_ctx* ctx, const std::vector<int>& ids, Group** out) {
    auto it = ctx->groups.find(ids);
    if (it != ctx->groups.end()) {
        it->second->last_use = ctx->clock;
        *out = it->second;
        return DBA_OK;
    }
    evict_groups(ctx);
    Group* g = new Group();
    g->last_use = ctx->clock;
    g->ids = ids;
    std::vector<Inst> hs;
    std::vector<Seg> segs;
    std::vector<InstSegs> isegs;
    for (size_t k = 0; k < ids.size(); k++) {
        Instance* in = ctx->inst[ids[k]];
        hs.push_back(in->h);
        g->total_tiles += in->h.nt;
        InstSegs r{(int32_t)segs.size(), 0};
        for (int t0 = 0; t0 < in->h.nt; t0 += kSegTiles) {
            segs.push_back(Seg{(int32_t)k, t0, std::min(kSegTiles, in->h.nt - t0), 0});
            r.count++;
        }
        isegs.push_back(r);
    }
    g->nseg = (int)segs.size();
    Instance* first = ctx->inst[ids[0]];
    if (ids.size() == 1 && g->nseg == 1) {
        g->solo_seg = first->h.seg;
        g->solo_rec = first->h.nbrec;
        g->solo_nt = first->h.nt;
    }
    g->model = first->p.model;
    g->tile = first->p.tile_x;
    g->tile_z = first->p.tile_z;
    g->threads = first->p.threads ? first->p.threads : default_threads(g->model, g->tile);
    g->dense_threads = first->p.threads ? first->p.threads : default_dense_threads(g->model, g->tile, g->total_tiles);
    g->conserved = ids.size() == 1 && first->p.mode == DBA_MODE_CONSERVED;
    for (int id : ids)
        if (!ctx->inst[id]->h.full_tiles) g->partial = true;
    // Column-march single-launch steps (ch_march_kernel): one large CH instance of
    // full 32 x 32 tiles, periodic both ways, not conserved; K tiles per strip,
    // the most that keep >= 1024 strips (measured: 2048^2 K = 4 18.4 us against
    // 20.8 at K = 2 and 22.5 at K = 8; 4096^2 K = 16 59.7 us, K = 8 60.2 us, K = 4
    // 63.1 us; 8192^2 K = 32 248.9 us against 253.0 at K = 8)
    g->nine = first->p.stencil != 5;
    if (ids.size() == 1 && g->model == DBA_MODEL_CH && g->tile == 32 && g->dense_threads == 256 &&
        first->p.mode != DBA_MODE_CONSERVED && first->h.full_tiles && first->p.bc_x == DBA_BC_PERIODIC &&
        first->p.bc_y == DBA_BC_PERIODIC && first->h.nt >= kMarchMinTiles) {
        for (int k : {32, 16, 8, 4, 2})
            if (first->h.nty % k == 0 && first->h.nt / k >= 1024) {
                g->march = k;
                break;
            }
    }
    // Resident steps: one CH or K93 instance (regular or DBA) whose tiles fit the chip at once
    if (ids.size() == 1 && first->p.mode != DBA_MODE_CONSERVED && first->p.threads == 0 &&
        (g->model == DBA_MODEL_CH || g->model == DBA_MODEL_DENDRITE_K93))
        resident_choose(ctx, g, first->h);
    // Speculative staging in single-launch K93 steps (k93_dense_kernel SPEC):
    // one instance of up to 1024 full 16 x 16 tiles at 512 threads (measured on
    // 512^2: 7.2 -> 6.7 us per step with the run-counter prefetch); larger grids
    // would pay the rings of both buffers of every sleeping tile in HBM bytes
    g->spec = ids.size() == 1 && g->model == DBA_MODEL_DENDRITE_K93 && g->tile == 16 && g->dense_threads == 512 &&
              first->h.full_tiles && first->h.nt <= 1024;
    // KH divides by dx, dy and the cell area; when all three are powers of two
    // (a power-of-two grid on the unit square) the step multiplies by their exact
    // reciprocals instead, which gives the same doubles (kh_cdiv in k_kh.h)
    if (g->model == DBA_MODEL_KH) {
        auto pow2 = [](double d) {
            int e = 0;
            return d > 0.0 && std::isfinite(d) && std::frexp(d, &e) == 0.5;
        };
        g->kh_p2 = true;
        for (int id : ids) {
            const Instance* in = ctx->inst.at(id);
            if (!(pow2(in->h.dx) && pow2(in->h.dy) && pow2(in->h.vol))) g->kh_p2 = false;
        }
    }
    // Model B: 65536 workgroups (4 blocks each on a fully awake 256^3 field)
    // measured faster than 16384 or 3072 with longer pipelines per wave. K94: the
    // waves that are resident at once (5 on each SIMD by registers), since a list is
    // mostly shorter and the dispatch of further ones costs: 256^3 dendrite, us per
    // step with 16, 20, 32, 64, 128 waves per CU: 22.3, 21.7, 22.4, 23.9, 27.0
    int64_t cap = g->model == DBA_MODEL_MODELB ? 65536 : (g->model == DBA_MODEL_DENDRITE_K94 ? 20 * ctx->n_cu : 4096);
    g->grid = (int)std::max<int64_t>(1, std::min<int64_t>(g->total_tiles, cap));
    // Model B column march (modelb_march_kernel, nz == 1: modelb_plane_kernel): one
    // instance, steps whose list is long enough. DBA_MODELB_SUPERBLOCKS set to a number
    // is the shortest list that takes it (0: none does); all give the same doubles. Layers
    // per strip: the fewest rounds of resident workgroups, each round 4 nl + 4 planes long.
    if (g->model == DBA_MODEL_MODELB && ids.size() == 1 && g->tile == 4) {
        const Inst& h = first->h;
        if (h.full_tiles && (h.nz > 1) == (g->tile_z == 4) && (int64_t)h.nx * h.ny < (1 << 28)) {
            const char* env = std::getenv("DBA_MODELB_SUPERBLOCKS");
            const std::string e = env ? env : "";
            g->mb_ntz = h.ntz;
            g->mb_ncx = (h.nx + MbMarch::TX - 1) / MbMarch::TX;
            g->mb_ncy = (h.ny + MbMarch::TY - 1) / MbMarch::TY;
            const int64_t cols = (int64_t)g->mb_ncx * g->mb_ncy, slots = (g->conserved ? 1 : 2) * (int64_t)ctx->n_cu;
            int64_t planes = INT64_MAX;
            for (int nl = 1; nl <= (g->conserved ? MbMarch::MLC : MbMarch::ML) && nl <= h.ntz; nl++) {
                const int64_t wgs = cols * ((h.ntz + nl - 1) / nl), cost = (wgs + slots - 1) / slots * (4 * nl + 4);
                if (cost < planes) {
                    planes = cost;
                    g->mb_nl = nl;
                }
            }
            // A plane of the march costs as much as about 1000 blocks of the block kernels
            // (conserved 550: one workgroup per CU). us per step, block kernels and march:
            // 64^3 30 and 32 (all 4096 awake); 128^3 (16 planes) 73 and 92 at 31% awake,
            // 105 and 95 at 62%; 160 x 160 x 100 (20) 84 and 110 at 30%, 123 and 112 at
            // 60%; 256^3 (136) 339 and 386 at 25%, 655 and 586 at 56%; conserved
            // 96 x 80 x 64 (12) 51 and 55 at 67%, 59 and 52 all awake. A list no grid of
            // this size can have: the march is not launched.
            // One plane: the block kernels fill 16 of a wave's 64 lanes and lose wherever
            // a march's workgroup has something to do (300^2 37 and 13, 43% awake 20 and
            // 12; 700^2 118 and 26, 25% awake 49 and 17); only on large grids with next to
            // nothing awake does its one workgroup per column cost more (2048^2 at 1% 63
            // and 42, 4096^2 at 0.6% 79 and 109, at 5% 214 and 122).
            int64_t from = h.nz > 1 ? planes * (g->conserved ? 550 : 1000) : (cols <= 8 * slots ? 1 : cols * 2 / 5);
            if (!e.empty() && e.find_first_not_of("0123456789") == std::string::npos) from = std::atoll(e.c_str());
            if (from > h.nt) from = 0;
            g->march_from = (int)from;
            // the block kernels then only take lists shorter than that, and return at once
            // from the others (160 x 160 x 100, all awake: 20000 workgroups 4 us more per
            // step than 5000; 30% awake: 71 us with 17000, 93 with 8500, 101 with 4250;
            // conserved 96 x 80 x 64, all awake: 58 with 6600 and 56.5 with 3300, 67%
            // awake 53 and 52, 59 with 1650)
            if (from > 0)
                g->grid = (int)std::max<int64_t>(1, std::min<int64_t>({g->grid, g->conserved ? (from + 1) / 2 : from, 12288}));
        }
    }
    size_t n = ids.size();
    HIP_TRY(hipMalloc(&g->d_insts, sizeof(Inst) * n));
    HIP_TRY(hipMemcpyAsync(g->d_insts, hs.data(), sizeof(Inst) * n, hipMemcpyHostToDevice, ctx->setup));
    size_t ns = segs.size();
    HIP_TRY(hipMalloc(&g->d_segs, sizeof(Seg) * ns));
    HIP_TRY(hipMemcpyAsync(g->d_segs, segs.data(), sizeof(Seg) * ns, hipMemcpyHostToDevice, ctx->setup));
    HIP_TRY(hipMalloc(&g->d_isegs, sizeof(InstSegs) * n));
    HIP_TRY(hipMemcpyAsync(g->d_isegs, isegs.data(), sizeof(InstSegs) * n, hipMemcpyHostToDevice, ctx->setup));
    // folded merges: as many segments as the kernels' offsets hold, and no instance
    // whose step needs the merged sums of the one before (a conserved shift, a CFL
    // time step). KH on 16 x 16 tiles keeps the merge launch: its kernel has no
    // registers left for the offsets (2048^2 at a fixed time step 164.6 us per step
    // with the merge launch, 168.2 folded; 8 x 8 tiles 26.4 and 24.8 us at 512^2)
    const bool three_d = g->model == DBA_MODEL_DENDRITE_K94 || g->model == DBA_MODEL_MODELB;
    g->fold = ns > 1 && ns <= (size_t)(three_d ? kFoldSegs : kFoldLanes) &&
              !(g->model == DBA_MODEL_KH && g->tile != 8);
    for (int id : ids) {
        const dba_params& p = ctx->inst.at(id)->p;
        if (p.mode == DBA_MODE_CONSERVED || (p.model == DBA_MODEL_KH && p.dt_mode == DBA_DT_CFL)) g->fold = false;
    }
    // two sets of partials (folded merges read one step's while the next one's are
    // written); counts padded with zeros to a whole scan
    const size_t nc = std::max<size_t>(ns, kFoldSegs);
    HIP_TRY(hipMalloc(&g->d_parts, sizeof(SegPart) * 2 * ns));
    HIP_TRY(hipMemsetAsync(g->d_parts, 0, sizeof(SegPart) * 2 * ns, ctx->setup));
    HIP_TRY(hipMalloc(&g->d_counts, sizeof(int32_t) * nc));
    HIP_TRY(hipMemsetAsync(g->d_counts, 0, sizeof(int32_t) * nc, ctx->setup));
    HIP_TRY(hipMalloc(&g->d_offsets, sizeof(int32_t) * (ns + 1)));
    HIP_TRY(hipMemsetAsync(g->d_offsets, 0, sizeof(int32_t) * (ns + 1), ctx->setup));
    std::vector<int32_t> dmap;
    if ((n > 1 || ns > 1) && (g->model == DBA_MODEL_CH || g->model == DBA_MODEL_DENDRITE_K93)) {
        // dense index -> instance << 24 | tile (groups hold at most 255 instances)
        bool fits = true;
        for (size_t k = 0; k < n; k++) fits = fits && hs[k].nt < (1 << 24);
        if (fits) {
            dmap.reserve((size_t)g->total_tiles);
            for (size_t k = 0; k < n; k++)
                for (int t = 0; t < hs[k].nt; t++) dmap.push_back((int32_t)((uint32_t)k << 24 | (uint32_t)t));
            HIP_TRY(hipMalloc(&g->d_dmap, sizeof(int32_t) * dmap.size()));
            HIP_TRY(hipMemcpyAsync(g->d_dmap, dmap.data(), sizeof(int32_t) * dmap.size(), hipMemcpyHostToDevice,
                                   ctx->setup));
        }
    }
    // the compute stream is used only after this host-side wait
    HIP_TRY(hipStreamSynchronize(ctx->setup));
    ctx->groups[ids] = g;
    *out = g;
    return DBA_OK;
}

// ---------------------------------------------------------------- launches

// Segment partials of step `step` of a run (folded merges alternate between two sets).
SegPart* parts_of(const Group* g, int step) { return g->d_parts + (g->fold && (step & 1) ? g->nseg : 0); }

WorkList wl_of(const Group* g) {
    return WorkList{g->d_insts, g->d_segs, g->d_offsets, g->nseg, g->solo_seg, g->solo_rec, g->solo_nt,
                    g->ids.size() == 1 ? 1 : 0, g->fold ? g->d_counts : nullptr};
}

template <int TB, int NT>
void launch_step_tb(const Group* g, hipStream_t s) {
    dim3 grid(g->grid), block(NT);
    switch (g->model) {
        case DBA_MODEL_CH: {
            // the strip layout needs NT <= TB*TB
            constexpr int NTC = NT <= TB * TB ? NT : TB * TB;
            if (g->partial)
                hipLaunchKernelGGL((ch_step_kernel<TB, NTC, true>), grid, dim3(NTC), 0, s, wl_of(g));
            else
                hipLaunchKernelGGL((ch_step_kernel<TB, NTC, false>), grid, dim3(NTC), 0, s, wl_of(g));
            break;
        }
        case DBA_MODEL_DENDRITE_K93:
            if (g->partial)
                hipLaunchKernelGGL((k93_step_kernel<TB, NT, true>), grid, block, 0, s, wl_of(g));
            else
                hipLaunchKernelGGL((k93_step_kernel<TB, NT, false>), grid, block, 0, s, wl_of(g));
            break;
        case DBA_MODEL_KH:
            // one thread per cell, whatever workgroup size the instance asks for
            // (it never changes results)
            if constexpr (TB <= 16) {
                if (g->kh_p2)
                    hipLaunchKernelGGL((kh_step_kernel<TB, true>), grid, dim3(TB * TB), 0, s, wl_of(g));
                else
                    hipLaunchKernelGGL((kh_step_kernel<TB, false>), grid, dim3(TB * TB), 0, s, wl_of(g));
            }
            break;
        default:
            break;
    }
}

template <int TB>
void launch_step_nt(const Group* g, hipStream_t s) {
    switch (g->threads) {
        case 64: launch_step_tb<TB, 64>(g, s); break;
        case 128: launch_step_tb<TB, 128>(g, s); break;
        case 512: launch_step_tb<TB, 512>(g, s); break;
        case 1024: launch_step_tb<TB, 1024>(g, s); break;
        default: launch_step_tb<TB, 256>(g, s); break;
    }
}

void launch_step(const Group* g, hipStream_t s) {
    if (g->model == DBA_MODEL_DENDRITE_K94 || g->model == DBA_MODEL_MODELB) {
        dim3 grid(g->grid), block(64);
        if (g->model == DBA_MODEL_MODELB) {
            // the march and the pair of block kernels: by list length, one of them
            // returns at once
            const int from = g->march_from > 0 ? g->march_from : INT_MAX;
            if (g->tile_z == 4) {
                if (g->march_from > 0) {
                    const int ntz = g->mb_ntz, ncol = g->mb_ncx * g->mb_ncy;
                    const dim3 mgrid((unsigned)(ncol * ((ntz + g->mb_nl - 1) / g->mb_nl)));
                    if (g->conserved)
                        hipLaunchKernelGGL(modelb_march_kernel<true>, mgrid, dim3(MbMarch::NT), 0, s, wl_of(g), from,
                                           g->mb_nl, g->mb_ncx, g->mb_ncy);
                    else
                        hipLaunchKernelGGL(modelb_march_kernel<false>, mgrid, dim3(MbMarch::NT), 0, s, wl_of(g), from,
                                           g->mb_nl, g->mb_ncx, g->mb_ncy);
                }
                if (g->march_from != 1) {
                    hipLaunchKernelGGL((modelb_mu_kernel<4, 4>), grid, block, 0, s, wl_of(g), from);
                    hipLaunchKernelGGL((modelb_update_kernel<4, 4>), grid, block, 0, s, wl_of(g), from);
                }
            } else {
                if (g->march_from > 0) {
                    const dim3 mgrid((unsigned)(g->mb_ncx * g->mb_ncy));
                    if (g->conserved)
                        hipLaunchKernelGGL(modelb_plane_kernel<true>, mgrid, dim3(MbMarch::NT), 0, s, wl_of(g), from,
                                           g->mb_ncx);
                    else
                        hipLaunchKernelGGL(modelb_plane_kernel<false>, mgrid, dim3(MbMarch::NT), 0, s, wl_of(g), from,
                                           g->mb_ncx);
                }
                if (g->march_from != 1) {
                    hipLaunchKernelGGL((modelb_mu_kernel<4, 1>), grid, block, 0, s, wl_of(g), from);
                    hipLaunchKernelGGL((modelb_update_kernel<4, 1>), grid, block, 0, s, wl_of(g), from);
                }
            }
        } else {
            // a wave per block; a multiple of 8 workgroups, so every XCD has as many
            const unsigned wgs = ((unsigned)(g->grid + 8 * kK94Waves - 1) / (8 * kK94Waves)) * 8;
            if (g->tile_z == 4)
                hipLaunchKernelGGL((k94_step_kernel<4, 4>), dim3(wgs), dim3(64 * kK94Waves), 0, s, wl_of(g));
            else
                hipLaunchKernelGGL((k94_step_kernel<4, 1>), dim3(wgs), dim3(64 * kK94Waves), 0, s, wl_of(g));
        }
        return;
    }
    switch (g->tile) {
        case 8: launch_step_nt<8>(g, s); break;
        case 16: launch_step_nt<16>(g, s); break;
        default: launch_step_nt<32>(g, s); break;
    }
}

// Single-launch steps: one instance in one segment (its whole state fits one
// canonicalising workgroup), a model with a single-launch kernel, no conserved
// shift (its per-step global sum needs the finalize).
// Conserved DBA needs the previous step's global change sum: single-launch
// steps recompute it in every workgroup, for one CH instance of <= 1024 tiles.
bool single_launch_params(const dba_params& p, int64_t nt) {
    if (p.mode == DBA_MODE_CONSERVED) return p.model == DBA_MODEL_CH && nt <= kSegTiles;
    return p.model == DBA_MODEL_CH || p.model == DBA_MODEL_DENDRITE_K93;
}

// Groups every instance of which is CH or K93 (one instance in one segment, or a
// tile map for the rest), conserved DBA only as one CH instance in one segment;
// batches only in mode 2, since every sleeping tile still takes a workgroup.
bool single_launch_ok(const dba_ctx* ctx, const Group* g) {
    if (ctx->single_launch == 0 || (ctx->single_launch == 1 && g->ids.size() != 1)) return false;
    if (!(g->ids.size() == 1 && g->nseg == 1) && !g->d_dmap) return false;
    for (int id : g->ids) {
        const Instance* in = ctx->inst.at(id);
        if (!single_launch_params(in->p, in->h.nt)) return false;
        if (in->p.mode == DBA_MODE_CONSERVED && !(g->ids.size() == 1 && g->nseg == 1)) return false;
    }
    return true;
}

template <int K>
void launch_march(const Group* g, hipStream_t s, int first, int step) {
    const dim3 grid((unsigned)(g->total_tiles / K));
    if (g->nine)
        hipLaunchKernelGGL((ch_march_kernel<K, true>), grid, dim3(256), 0, s, g->d_insts, first, step);
    else
        hipLaunchKernelGGL((ch_march_kernel<K, false>), grid, dim3(256), 0, s, g->d_insts, first, step);
}

template <int TB, int NT>
void launch_dense_tb(const Group* g, hipStream_t s, int first, int step) {
    const dim3 grid((unsigned)g->total_tiles);
    if (g->model == DBA_MODEL_CH) {
        constexpr int NTC = NT <= TB * TB ? NT : TB * TB;
        if (g->conserved && g->partial)
            hipLaunchKernelGGL((ch_dense_kernel<TB, NTC, true, true>), grid, dim3(NTC), 0, s, g->d_insts, g->d_dmap,
                               first, step);
        else if (g->conserved)
            hipLaunchKernelGGL((ch_dense_kernel<TB, NTC, true, false>), grid, dim3(NTC), 0, s, g->d_insts, g->d_dmap,
                               first, step);
        else if (g->partial)
            hipLaunchKernelGGL((ch_dense_kernel<TB, NTC, false, true>), grid, dim3(NTC), 0, s, g->d_insts, g->d_dmap,
                               first, step);
        else
            hipLaunchKernelGGL((ch_dense_kernel<TB, NTC, false, false>), grid, dim3(NTC), 0, s, g->d_insts,
                               g->d_dmap, first, step);
    } else if (g->partial) {
        hipLaunchKernelGGL((k93_dense_kernel<TB, NT, true>), grid, dim3(NT), 0, s, g->d_insts, g->d_dmap, first,
                           step);
    } else if (TB == 16 && NT == 512 && g->spec) {
        hipLaunchKernelGGL((k93_dense_kernel<16, 512, false, true>), grid, dim3(512), 0, s, g->d_insts, g->d_dmap,
                           first, step);
    } else {
        hipLaunchKernelGGL((k93_dense_kernel<TB, NT, false>), grid, dim3(NT), 0, s, g->d_insts, g->d_dmap, first,
                           step);
    }
}

template <int TB>
void launch_dense_nt(const Group* g, hipStream_t s, int first, int step) {
    switch (g->dense_threads) {
        case 64: launch_dense_tb<TB, 64>(g, s, first, step); break;
        case 128: launch_dense_tb<TB, 128>(g, s, first, step); break;
        case 512: launch_dense_tb<TB, 512>(g, s, first, step); break;
        case 1024: launch_dense_tb<TB, 1024>(g, s, first, step); break;
        default: launch_dense_tb<TB, 256>(g, s, first, step); break;
    }
}

void launch_dense(const Group* g, hipStream_t s, int first, int step) {
    if (g->march) {
        switch (g->march) {
            case 32: launch_march<32>(g, s, first, step); break;
            case 16: launch_march<16>(g, s, first, step); break;
            case 8: launch_march<8>(g, s, first, step); break;
            case 4: launch_march<4>(g, s, first, step); break;
            default: launch_march<2>(g, s, first, step); break;
        }
        return;
    }
    switch (g->tile) {
        case 8: launch_dense_nt<8>(g, s, first, step); break;
        case 16: launch_dense_nt<16>(g, s, first, step); break;
        default: launch_dense_nt<32>(g, s, first, step); break;
    }
}

// The end of step `step` of a run (rotate), or the rebuilt worklists of the current
// awake sets. last: no step follows, so the instance sums are merged here.
void launch_finalize(const Group* g, hipStream_t s, int rotate, int step, bool last) {
    SegPart* parts = parts_of(g, step);
    const SegPart* pend = g->fold && rotate && step > 0 ? parts_of(g, step - 1) : nullptr;
    const int n_inst = (int)g->ids.size();
    const unsigned per_inst = (unsigned)((n_inst + kFinNT / 64 - 1) / (kFinNT / 64));  // workgroups, a wave per instance
    hipLaunchKernelGGL(finalize_kernel, dim3((unsigned)g->nseg + (pend ? per_inst : 0u)), dim3(kFinNT), 0, s,
                       g->d_insts, g->d_segs, g->nseg, parts, g->d_counts, g->d_offsets, rotate, n_inst == 1 ? 1 : 0,
                       pend, g->d_isegs, n_inst);
    if (g->nseg > 1 && (!g->fold || last)) {
        // workgroup 0 scans the segment counts; the others reduce 16 instances each
        const unsigned wgs = 1u + per_inst;
        hipLaunchKernelGGL(finalize_merge_kernel, dim3(wgs), dim3(kFinNT), 0, s, g->d_insts, g->nseg, g->d_isegs,
                           n_inst, parts, g->d_counts, g->d_offsets, rotate);
    }
}

hipEvent_t pooled_event(dba_ctx* ctx) {
    hipEvent_t e = nullptr;
    if (!ctx->ev_pool.empty()) {
        e = ctx->ev_pool.back();
        ctx->ev_pool.pop_back();
    } else {
        (void)hipEventCreate(&e);
    }
    ctx->ev_used.push_back(e);
    return e;
}

dba_status partition(dba_ctx* ctx, const int32_t* ids, int32_t n_ids, std::vector<std::vector<int>>* parts) {
    if (n_ids <= 0 || !ids) return fail(DBA_ERR_INVALID, "no instances given");
    std::vector<int> seen;
    for (int k = 0; k < n_ids; k++) {
        int id = ids[k];
        auto it = ctx->inst.find(id);
        if (it == ctx->inst.end()) return fail(DBA_ERR_NOTFOUND, "unknown instance %d", id);
        if (std::find(seen.begin(), seen.end(), id) != seen.end())
            return fail(DBA_ERR_INVALID, "instance %d listed twice", id);
        seen.push_back(id);
        const dba_params& p = it->second->p;
        int thr = p.threads ? p.threads : default_threads(p.model, p.tile_x);
        bool placed = false;
        for (auto& part : *parts) {
            const dba_params& q = ctx->inst[part[0]]->p;
            int thq = q.threads ? q.threads : default_threads(q.model, q.tile_x);
            if (q.model == p.model && q.tile_x == p.tile_x && q.tile_z == p.tile_z && thq == thr &&
                part.size() < 255) {
                part.push_back(id);
                placed = true;
                break;
            }
        }
        if (!placed) parts->push_back({id});
    }
    return DBA_OK;
}

// The state-restoring launches after n_steps single-launch or resident steps.
dba_status launch_canon(dba_ctx* ctx, const Group* g, int n_steps, uint32_t* res = nullptr) {
    if (!g->d_dmap) {
        hipLaunchKernelGGL(dense_canon_kernel, dim3(1), dim3(kFinNT), 0, ctx->stream, g->d_insts, n_steps, res);
    } else {
        hipLaunchKernelGGL(dense_canon_seg_kernel, dim3((unsigned)g->nseg), dim3(kFinNT), 0, ctx->stream, g->d_insts,
                           g->d_segs, g->d_parts, g->d_counts, n_steps, (const uint32_t*)res);
        LAUNCH_CHECK();
        hipLaunchKernelGGL(dense_canon_merge_kernel, dim3(1), dim3(kFinNT), 0, ctx->stream, g->d_insts, g->d_isegs,
                           (int)g->ids.size(), g->d_parts, g->d_counts, n_steps, res);
    }
    LAUNCH_CHECK();
    return DBA_OK;
}

// ---- resident steps (k_resident.h)

// The cooperative launch costs about 15 us more than the launches it replaces have
// around them (256^2: 41 us + 2.7 us per step against 28 + 4.4; 1024^2: 54 + 4.4
// against 36 + 7.0), so calls of fewer steps keep single-launch steps.
constexpr int kResidentMinSteps = 12;

template <int TB, int NT>
const void* ch_resident_fn(bool nine) {
    return nine ? (const void*)ch_resident_kernel<TB, NT, true> : (const void*)ch_resident_kernel<TB, NT, false>;
}

// The kernel of a group's tile: `per_tile` threads on each tile (K93: one per cell).
const void* resident_kernel(const Group* g, int per_tile) {
    if (g->model == DBA_MODEL_DENDRITE_K93) switch (g->tile) {
            case 8: return (const void*)k93_resident_kernel<8>;
            case 16: return (const void*)k93_resident_kernel<16>;
            default: return (const void*)k93_resident_kernel<32>;
        }
    switch (g->tile) {
        case 8: return ch_resident_fn<8, 64>(g->nine);
        case 16: return ch_resident_fn<16, 128>(g->nine);
        default: return per_tile == 1024 ? ch_resident_fn<32, 1024>(g->nine) : ch_resident_fn<32, 256>(g->nine);
    }
}

size_t resident_bytes(const Group* g, int w, int h) {
    return g->model == DBA_MODEL_DENDRITE_K93 ? k93_resident_bytes(w, h) : ch_resident_bytes(w, h);
}

// Whether `wgs` workgroups of the kernel are certainly resident at once. The
// occupancy the runtime computes does not count the scalar registers the trap
// handler takes from every wave (measured: 28 one-wave workgroups per CU promised,
// 24 resident), so at most 24 waves per CU; and a sixteenth is kept free where
// several share a CU (27 promised by their LDS, 26.7 resident).
bool all_resident(const dba_ctx* ctx, const void* f, int threads, size_t lds, int64_t wgs) {
    constexpr size_t kLdsPerCu = 160 * 1024, kMostLds = kLdsPerCu - 2048;  // (less the kernels' static LDS)
    if (lds > kMostLds) return false;
    // the most any shape asks for, since the attribute is the function's: a smaller
    // instance's bytes would lower it below what a larger one launches with
    if (lds > 64 * 1024 && hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMostLds) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    int blocks = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, f, threads, lds) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    blocks = std::min(blocks, 24 / (threads / 64));
    const int64_t all = (int64_t)blocks * ctx->n_cu;
    return wgs <= (blocks > 1 ? all - all / 16 : all);
}

// Region and workgroup of a CH group's resident steps, if the grid fits the chip.
void resident_choose(const dba_ctx* ctx, Group* g, const Inst& h) {
    int coop = 0;
    if (hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, ctx->device) != hipSuccess || !coop) return;
    struct Shape {
        int gx, gy, threads, per_tile;
    };
    // smallest regions first: per step a region waits for one exchange whatever its
    // size, so a grid that leaves room takes more threads per cell, and a larger one
    // larger regions (fewer frames). us per step over 1000 steps, single-launch
    // steps -> this: 32 x 32 tiles 256^2 4.4 -> 2.7 (512 or 1024 threads per tile; 256: 3.5),
    // 1024^2 7.1 -> 4.4 (one tile per workgroup: 7.0, two: 7.1), 1200 x 1100
    // 15.2 -> 6.2, 1571 x 1390 15.8 -> 7.7; 16 x 16 tiles 512^2 4.5 -> 2.6, 1024^2 8.4 -> 5.0; 8 x 8 tiles
    // 512^2 5.7 -> 3.1
    std::vector<Shape> shapes = {{1, 1, 1024, 1024}, {2, 2, 1024, 256}, {3, 2, 768, 256}, {3, 3, 1024, 256}};
    if (g->tile == 16) shapes = {{2, 2, 512, 128}, {4, 4, 1024, 128}};
    if (g->tile == 8) shapes = {{4, 2, 512, 64}, {4, 4, 1024, 64}};
    // K93: one cell per thread. Several cells per thread (4 x 4 tiles of 16 x 16) make a
    // larger grid fit, but one dendrite's awake tiles then crowd on few CUs: 1000^2
    // 16.5 us per step against 7.9. Smaller regions with several on a CU exchange more:
    // 512^2 4.3 - 5.2 against 4.0. us per step over 1000 steps, single-launch steps ->
    // this: 16 x 16 tiles 256^2 4.9 -> 3.5, 512^2 5.8 -> 4.0 (regular mode 9.2 -> 3.4);
    // 8 x 8 tiles 512^2 6.9 -> 4.4; 32 x 32 tiles 512^2 7.6 -> 4.2
    if (g->model == DBA_MODEL_DENDRITE_K93) {
        shapes = {{1, 1, 1024, 1024}};
        if (g->tile == 16) shapes = {{1, 1, 256, 256}, {2, 2, 1024, 256}};
        if (g->tile == 8) shapes = {{2, 2, 256, 64}, {4, 4, 1024, 64}};
    }
    for (const Shape& s : shapes) {
        const void* f = resident_kernel(g, s.per_tile);
        const size_t lds = resident_bytes(g, g->tile * s.gx, g->tile * s.gy);
        const int64_t wgs = (int64_t)((h.ntx + s.gx - 1) / s.gx) * ((h.nty + s.gy - 1) / s.gy);
        if (s.threads < ch_resident_threads(g->tile * s.gx, g->tile * s.gy)) continue;
        if (!all_resident(ctx, f, s.threads, lds, wgs)) continue;
        g->res_gx = s.gx;
        g->res_gy = s.gy;
        g->res_threads = s.threads;
        g->res_per_tile = s.per_tile;
        return;
    }
}

// The exchange buffer of `words`, cleared when the sequence numbers start over.
bool resident_buffer(dba_ctx* ctx, size_t words, int n_steps) {
    if (!ctx->stuck) {
        if (hipHostMalloc((void**)&ctx->stuck, sizeof(int)) != hipSuccess) return false;
        *ctx->stuck = 0;
    }
    const bool wrap = ctx->xseq > 0xffffffffu - (uint32_t)n_steps - 2u;
    if (words <= ctx->xwords && !wrap) return true;
    if (hipStreamSynchronize(ctx->stream) != hipSuccess) return false;
    if (words > ctx->xwords) {
        if (ctx->xbuf) (void)hipFree(ctx->xbuf);
        ctx->xbuf = nullptr;
        ctx->xwords = 0;
        if (hipMalloc(&ctx->xbuf, sizeof(ResHead) + words * sizeof(uint64_t)) != hipSuccess) {
            ctx->xbuf = nullptr;
            return false;
        }
        // (a launch given up before this that the host has not taken notice of)
        const ResHead head{*(volatile int*)ctx->stuck ? kResGivenUp : kResRunning, 0, ctx->stuck, {}};
        if (hipMemcpy(ctx->xbuf, &head, sizeof(head), hipMemcpyHostToDevice) != hipSuccess) return false;
        ctx->xwords = words;
    }
    ctx->xseq = 1;
    return hipMemsetAsync(ctx->xbuf + 1, 0, ctx->xwords * sizeof(uint64_t), ctx->stream) == hipSuccess;
}

// The process's contexts on a device, after adding `d`. A context alone on its device
// takes resident launches. Where there are others it does not: of two such launches,
// each half resident, both would be given up, and single-launch steps of two contexts
// overlap, so they finish sooner than resident ones after each other (two contexts of
// 1024^2, 2000 steps: 18.5 ms against 22).
int live_contexts(int device, int d) {
    static std::mutex m;
    static std::map<int, int>* live = new std::map<int, int>();  // kept until the process ends
    std::lock_guard<std::mutex> lock(m);
    return (*live)[device] += d;
}

// Whether an instance has resident launches that the host has not waited for.
bool is_unsettled(const dba_ctx* ctx, int id) {
    return std::find(ctx->unsettled.begin(), ctx->unsettled.end(), id) != ctx->unsettled.end();
}

// n_steps of one group as a resident launch and its canonicalising kernels; *taken is
// false where the launch could not be had (the other paths need less) or must not be.
dba_status enqueue_resident(dba_ctx* ctx, Group* g, int n_steps, bool* taken) {
    *taken = false;
    if (!g->res_gx || !ctx->resident || ctx->single_launch == 0 || ctx->timing || n_steps < kResidentMinSteps)
        return DBA_OK;
    if (live_contexts(ctx->device, 0) > 1) return DBA_OK;
    const int h_id = g->ids[0];
    const Inst& h = ctx->inst.at(h_id)->h;
    const int nt = h.nt, gx = g->res_gx, gy = g->res_gy;
    const unsigned wgs = (unsigned)(((h.ntx + gx - 1) / gx) * ((h.nty + gy - 1) / gy));
    const int slots = frame_slots(gx * g->tile, gy * g->tile);
    const size_t flags = 2 * (size_t)nt;
    const int fields = g->model == DBA_MODEL_DENDRITE_K93 ? 2 : 1;
    const size_t words = 2 * (size_t)wgs * (size_t)slots * 2 * fields + flags;
    const bool have = resident_buffer(ctx, words, n_steps);
    hipError_t e = hipErrorOutOfMemory;
    if (have) {
        const void* f = resident_kernel(g, g->res_per_tile);
        const size_t lds = resident_bytes(g, gx * g->tile, gy * g->tile);
        uint64_t* frames = (uint64_t*)(ctx->xbuf + 1);
        Exchange X{frames, frames + (words - flags), ctx->wait_polls, ctx->xseq, slots};
        const Inst* insts = g->d_insts;
        int n = n_steps, ax = gx, ay = gy;
        void* args[] = {(void*)&insts, (void*)&X, (void*)&n, (void*)&ax, (void*)&ay};
        e = hipLaunchCooperativeKernel(f, dim3(wgs), dim3((unsigned)g->res_threads), args, (unsigned)lds, ctx->stream);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        // too little memory is tried again; another process may have the GPU's queue for
        // cooperative launches, and every attempt to get it takes 15 ms
        if (e == hipErrorCooperativeLaunchTooLarge) g->res_gx = 0;
        else if (have) ctx->resident = false;
        return DBA_OK;
    }
    ctx->xseq += (uint32_t)n_steps + 1u;
    ctx->resident_calls++;
    if (!is_unsettled(ctx, h_id)) ctx->unsettled.push_back(h_id);
    *taken = true;
    return launch_canon(ctx, g, n_steps, &ctx->xbuf->state);
}

dba_status enqueue_steps(dba_ctx* ctx, const std::vector<Group*>& gs, int n_steps, bool timed) {
    // single-launch groups: n steps, then one canonicalisation
    for (Group* g : gs) {
        if (n_steps == 0 || !single_launch_ok(ctx, g)) continue;
        for (int s = 0; s < n_steps + 1; s++) {
            hipEvent_t a = nullptr, b = nullptr;
            if (timed) {
                a = pooled_event(ctx);
                b = pooled_event(ctx);
                (void)hipEventRecord(a, ctx->stream);
            }
            if (s < n_steps) {
                launch_dense(g, ctx->stream, s == 0, s);
            } else {
                const dba_status st = launch_canon(ctx, g, n_steps);
                if (st != DBA_OK) return st;
            }
            LAUNCH_CHECK();
            if (timed) {
                (void)hipEventRecord(b, ctx->stream);
                (s < n_steps ? ctx->ev_step : ctx->ev_fin).push_back({a, b});
            }
        }
    }
    for (int s = 0; s < n_steps; s++) {
        for (Group* g : gs) {
            if (single_launch_ok(ctx, g)) continue;
            hipEvent_t a = nullptr, b = nullptr, c = nullptr;
            if (timed) {
                a = pooled_event(ctx);
                b = pooled_event(ctx);
                c = pooled_event(ctx);
                (void)hipEventRecord(a, ctx->stream);
            }
            launch_step(g, ctx->stream);
            LAUNCH_CHECK();
            if (timed) (void)hipEventRecord(b, ctx->stream);
            launch_finalize(g, ctx->stream, 1, s, s + 1 == n_steps);
            LAUNCH_CHECK();
            if (timed) {
                (void)hipEventRecord(c, ctx->stream);
                ctx->ev_step.push_back({a, b});
                ctx->ev_fin.push_back({b, c});
            }
        }
    }
    return DBA_OK;
}

dba_status prepare_groups(dba_ctx* ctx, const int32_t* ids, int32_t n_ids, std::vector<Group*>* gs) {
    std::vector<std::vector<int>> parts;
    dba_status st = partition(ctx, ids, n_ids, &parts);
    if (st != DBA_OK) return st;
    ctx->clock++;
    for (int k = 0; k < n_ids; k++) ctx->inst[ids[k]]->stepped = true;
    for (auto& part : parts) {
        Group* g = nullptr;
        st = get_group(ctx, part, &g);
        if (st != DBA_OK) return st;
        gs->push_back(g);
    }
    // KH instances whose state was uploaded since their last step
    for (int k = 0; k < n_ids; k++) {
        Instance* in = ctx->inst[ids[k]];
        if (in->needs_prime) {
            st = kh_prime(ctx, in);
            if (st != DBA_OK) return st;
        }
    }
    // (re)build the worklists from the current awake sets
    for (Group* g : *gs) {
        launch_finalize(g, ctx->stream, 0, 0, true);
        LAUNCH_CHECK();
    }
    return DBA_OK;
}

Instance* find(dba_ctx* ctx, int id) {
    auto it = ctx->inst.find(id);
    return it == ctx->inst.end() ? nullptr : it->second;
}

dba_status ensure_staging(dba_ctx* ctx, size_t n) {
    if (ctx->staging_n >= n) return DBA_OK;
    if (ctx->staging) (void)hipFree(ctx->staging);
    ctx->staging = nullptr;
    ctx->staging_n = 0;
    HIP_TRY(hipMalloc(&ctx->staging, n * sizeof(double)));
    ctx->staging_n = n;
    return DBA_OK;
}

}  // namespace

namespace {
// Waits for the compute stream. Steps of resident launches that were given up are then
// made on the other paths, so the caller never sees them missing; *redone says so to
// calls that had already read the state. The context keeps to the other paths after
// that: what held the launch up (another process on the GPU) may still be there.
dba_status wait_stream(dba_ctx* ctx, bool* redone = nullptr) {
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    std::vector<int> ids;
    ids.swap(ctx->unsettled);
    if (!ctx->stuck || !*(volatile int*)ctx->stuck) return DBA_OK;
    *ctx->stuck = 0;
    ctx->resident = false;
    HIP_TRY(hipMemsetAsync(ctx->xbuf, 0, 2 * sizeof(uint32_t), ctx->stream));  // (not the stuck pointer)
    for (int id : ids) {
        Instance* in = ctx->inst.at(id);
        int64_t ctr[4];
        HIP_TRY(hipMemcpy(ctr, in->h.ctr, sizeof(ctr), hipMemcpyDeviceToHost));
        if (ctr[3] == 0) continue;
        HIP_TRY(hipMemsetAsync(in->h.ctr + 3, 0, sizeof(int64_t), ctx->stream));
        // (the launch counted in the history of its steps as it went)
        if (ctr[0] < in->h.hist_cap)
            HIP_TRY(hipMemsetAsync(in->h.hist + 2 * ctr[0], 0, sizeof(int32_t) * 2 * (size_t)(in->h.hist_cap - ctr[0]),
                                   ctx->stream));
        std::vector<Group*> gs;
        const int32_t one = id;
        dba_status st = prepare_groups(ctx, &one, 1, &gs);
        for (int64_t left = ctr[3]; st == DBA_OK && left > 0;) {
            const int n = (int)std::min<int64_t>(left, 1 << 16);
            st = enqueue_steps(ctx, gs, n, false);
            left -= n;
        }
        if (st != DBA_OK) return st;
        ctx->resident_redone += ctr[3];
        if (redone) *redone = true;
    }
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    return DBA_OK;
}

// Before work on an instance that a redone step must not come after.
dba_status settle(dba_ctx* ctx, int id, bool* redone = nullptr) {
    return is_unsettled(ctx, id) ? wait_stream(ctx, redone) : DBA_OK;
}

// ... of a step call: the groups anew if steps were redone.
dba_status settle_groups(dba_ctx* ctx, const int32_t* ids, int32_t n_ids, std::vector<Group*>* gs) {
    bool redone = false;
    for (int k = 0; k < n_ids; k++) {
        const dba_status st = settle(ctx, ids[k], &redone);
        if (st != DBA_OK) return st;
    }
    if (!redone) return DBA_OK;
    gs->clear();
    return prepare_groups(ctx, ids, n_ids, gs);
}
}  // namespace

#define DBA_TRY(expr)                                 \
    do {                                              \
        const dba_status t_ = (expr);                 \
        if (t_ != DBA_OK) return t_;                  \
    } while (0)

#define WAIT_STREAM(ctx) DBA_TRY(wait_stream(ctx))

// ... after the state was read on the stream: `again` (the same call) if steps were redone
#define WAIT_READ(ctx, again)                         \
    do {                                              \
        bool redone_ = false;                         \
        DBA_TRY(wait_stream(ctx, &redone_));          \
        if (redone_) return again;                    \
    } while (0)

// ===================================================================== C ABI

namespace {
// Device scratch of one droplet analysis, freed when the call returns.
struct CcScratch {
    std::vector<void*> ptrs;
    ~CcScratch() {
        for (void* q : ptrs) (void)hipFree(q);
    }
    template <typename T>
    hipError_t get(T** out, size_t count) {
        void* q = nullptr;
        const hipError_t e = hipMalloc(&q, sizeof(T) * (count ? count : 1));
        if (e == hipSuccess) ptrs.push_back(q);
        *out = (T*)q;
        return e;
    }
};
}  // namespace

extern "C" {

const char* dba_last_error(void) { return g_error.c_str(); }

dba_status dba_init(int32_t device, dba_ctx** out) {
    if (!out) return fail(DBA_ERR_INVALID, "out is null");
    int n = 0;
    HIP_TRY(hipGetDeviceCount(&n));
    if (device < 0 || device >= n) return fail(DBA_ERR_INVALID, "device %d not present (%d devices)", device, n);
    HIP_TRY(hipSetDevice(device));
    dba_ctx* ctx = new dba_ctx();
    ctx->device = device;
    hipError_t e = hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        delete ctx;
        return fail(DBA_ERR_HIP, "hipStreamCreate failed: %s", hipGetErrorString(e));
    }
    e = hipStreamCreateWithFlags(&ctx->setup, hipStreamNonBlocking);
    if (e != hipSuccess) {
        (void)hipStreamDestroy(ctx->stream);
        delete ctx;
        return fail(DBA_ERR_HIP, "hipStreamCreate failed: %s", hipGetErrorString(e));
    }
    void* sp = nullptr;
    e = hipGetSymbolAddress(&sp, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !sp) {
        (void)hipStreamDestroy(ctx->stream);
        (void)hipStreamDestroy(ctx->setup);
        delete ctx;
        return fail(DBA_ERR_HIP, "hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
    }
    ctx->scratch = (unsigned char*)sp;
    int cu = 0;
    if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && cu > 0)
        ctx->n_cu = cu;
    HIP_TRY(hipMalloc(&ctx->d_flag, sizeof(int)));
    HIP_TRY(hipMalloc(&ctx->d_diag, sizeof(double) * (3 * kDiagBlocks + kMaxFrontCols + 8)));
    HIP_TRY(hipMalloc(&ctx->d_cols, sizeof(int32_t) * kMaxFrontCols));
    for (auto& m : ctx->markers) HIP_TRY(hipEventCreate(&m));
    live_contexts(device, 1);
    *out = ctx;
    return DBA_OK;
}

dba_status dba_finalize(dba_ctx* ctx) {
    if (!ctx) return DBA_OK;
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
    live_contexts(ctx->device, -1);
    std::vector<int> ids;
    for (auto& kv : ctx->inst) ids.push_back(kv.first);
    for (int id : ids) dba_instance_destroy(ctx, id);
    for (auto& kv : ctx->graphs) (void)hipGraphExecDestroy(kv.second.exec);
    for (auto e : ctx->ev_used) (void)hipEventDestroy(e);
    for (auto e : ctx->ev_pool) (void)hipEventDestroy(e);
    for (auto m : ctx->markers) (void)hipEventDestroy(m);
    if (ctx->staging) (void)hipFree(ctx->staging);
    if (ctx->xbuf) (void)hipFree(ctx->xbuf);
    if (ctx->stuck) (void)hipHostFree(ctx->stuck);
    if (ctx->d_flag) (void)hipFree(ctx->d_flag);
    if (ctx->d_diag) (void)hipFree(ctx->d_diag);
    if (ctx->d_cols) (void)hipFree(ctx->d_cols);
    (void)hipStreamDestroy(ctx->stream);
    (void)hipStreamDestroy(ctx->setup);
    delete ctx;
    return DBA_OK;
}

dba_status dba_footprint(const dba_params* p, int64_t* bytes) {
    if (!p || !bytes) return fail(DBA_ERR_INVALID, "null argument");
    dba_status st = validate(*p);
    if (st != DBA_OK) return st;
    *bytes = footprint_of(*p);
    return DBA_OK;
}

dba_status dba_device_memory(dba_ctx* ctx, int64_t* free_bytes, int64_t* total_bytes) {
    if (!ctx || !free_bytes || !total_bytes) return fail(DBA_ERR_INVALID, "null argument");
    HIP_TRY(hipSetDevice(ctx->device));
    size_t f = 0, t = 0;
    HIP_TRY(hipMemGetInfo(&f, &t));
    *free_bytes = (int64_t)f;
    *total_bytes = (int64_t)t;
    return DBA_OK;
}

dba_status dba_instance_create(dba_ctx* ctx, const dba_params* pp, int32_t* id) {
    if (!ctx || !pp || !id) return fail(DBA_ERR_INVALID, "null argument");
    dba_status st = validate(*pp);
    if (st != DBA_OK) return st;
    HIP_TRY(hipSetDevice(ctx->device));
    Instance* in = new Instance();
    in->p = *pp;
    if (in->p.tile_z <= 0) in->p.tile_z = 1;
    const dba_params& p = in->p;
    Layout L = layout_of(p);
    Inst& h = in->h;
    memset(&h, 0, sizeof(h));
    h.model = p.model;
    h.mode = p.mode;
    h.nx = p.nx; h.ny = p.ny; h.nz = p.nz;
    h.tx = p.tile_x; h.ty = p.tile_y; h.tz = p.tile_z;
    h.ntx = L.ntx; h.nty = L.nty; h.ntz = L.ntz; h.nt = L.nt; h.nwords = L.nwords;
    h.bc_x = p.bc_x; h.bc_y = p.bc_y; h.bc_z = p.bc_z;
    h.stencil = p.stencil; h.aniso_j = p.aniso_j; h.dt_mode = p.dt_mode; h.metric_kind = p.metric_kind;
    h.nsets = L.nsets;
    h.nfields = L.nf;
    h.ncons = 0;
    if (p.mode == DBA_MODE_CONSERVED) {
        if (p.model == DBA_MODEL_CH) h.ncons = 1;
        if (p.model == DBA_MODEL_KH) h.ncons = 4;
        if (p.model == DBA_MODEL_MODELB) h.ncons = 3;
    }
    for (int f = 0; f < kMaxFields; f++) h.field_set[f] = 0;
    if (L.nsets == 2) h.field_set[1] = 1;
    h.full_tiles = (p.nx % p.tile_x == 0 && p.ny % p.tile_y == 0 && p.nz % p.tile_z == 0) ? 1 : 0;
    h.dx = p.dx; h.dy = p.dy > 0 ? p.dy : p.dx; h.dz = p.dz > 0 ? p.dz : p.dx; h.dt = p.dt;
    h.thresh_a = p.thresh_a; h.thresh_b = p.thresh_b;
    h.ntotal = (double)L.n;
    derive_constants(p, h);
    h.tau = p.tau; h.eps_bar = p.eps_bar; h.delta = p.delta; h.alpha = p.alpha; h.gamma = p.gamma;
    h.theta0 = p.theta0; h.latent_k = p.latent_k; h.t_eq = p.t_eq;
    h.mobility = p.mobility; h.kappa = p.kappa; h.react_gamma = p.react_gamma; h.cbar = p.cbar;
    h.chi_xy = p.chi_xy; h.chi_xz = p.chi_xz; h.chi_yz = p.chi_yz;
    h.chi_xb = p.chi_xb; h.chi_yb = p.chi_yb; h.chi_zb = p.chi_zb;
    h.v_x = p.v_x; h.v_y = p.v_y; h.v_z = p.v_z; h.r_x = p.r_x; h.r_y = p.r_y; h.r_z = p.r_z;
    h.n_exp = p.n_exp; h.m_exp = p.m_exp;
    h.epsx_sq = p.epsx_sq; h.epsy_sq = p.epsy_sq; h.epsz_sq = p.epsz_sq; h.epsphi_sq = p.epsphi_sq;
    h.mob_x = p.mob_x; h.mob_y = p.mob_y; h.mob_z = p.mob_z; h.mob_phi = p.mob_phi;
    h.k_eq = p.k_eq; h.z_crit = p.z_crit; h.p_gel = p.p_gel; h.k_0 = p.k_0;
    h.gas_gamma = p.gas_gamma; h.cfl = p.cfl; h.vol = h.dx * h.dy;
    h.hist_cap = std::max(0, p.history_cap);

    Arena arena;
    for (int f = 0; f < L.nf; f++) {
        arena.add(&h.buf[0][f], (size_t)L.n);
        arena.add(&h.buf[1][f], (size_t)L.n);
    }
    for (int a = 0; a < L.naux; a++) arena.add(&h.aux[a], (size_t)L.aux_len);
    for (int s = 0; s < 2; s++) {
        arena.add(&h.a_cur[s], (size_t)L.nwords);
        arena.add(&h.nflag[s], (size_t)L.nt);
        arena.add(&h.par[s], (size_t)L.nwords);
        arena.add(&h.dF[s], (size_t)L.nsets * L.nt);
        arena.add(&h.dP[s], (size_t)L.nsets * L.nt);
    }
    arena.add(&h.druns, (size_t)L.nt);
    arena.add(&h.tpart, (size_t)kMaxFields * L.nt);
    arena.add(&h.tspeed, (size_t)2 * L.nt);
    arena.add(&h.s_tile, (size_t)kMaxFields * 2 * L.nt);
    arena.add(&h.scal, 16);
    arena.add(&h.ctr, 4);
    arena.add(&h.hist, (size_t)2 * h.hist_cap + 2);
    arena.add(&h.seg, (size_t)L.nt);
    arena.add(&h.nbrec, (size_t)L.nt);
    arena.add(&in->d_self, 1);
    st = alloc_arena(in, arena, ctx->setup);
    if (st != DBA_OK) {
        free_instance(in);
        delete in;
        return st;
    }
    // all tiles awake at start (example_Dendritic_growth/kernel.cu:149-161)
    std::vector<uint64_t> all((size_t)L.nwords, ~0ull);
    if (L.nt % 64) all.back() = (1ull << (L.nt % 64)) - 1ull;
    double scal[16] = {0};
    scal[1] = p.dt;
    for (int s = 0; s < L.nsets; s++)
        HIP_TRY(hipMemcpyAsync(h.a_cur[s], all.data(), sizeof(uint64_t) * L.nwords, hipMemcpyHostToDevice,
                               ctx->setup));
    HIP_TRY(hipMemcpyAsync(h.scal, scal, sizeof(scal), hipMemcpyHostToDevice, ctx->setup));
    HIP_TRY(hipMemcpyAsync(in->d_self, &h, sizeof(Inst), hipMemcpyHostToDevice, ctx->setup));
    // set-up lands before any later work on the compute stream (host-side wait);
    // work already running there for other instances is not waited for
    HIP_TRY(hipStreamSynchronize(ctx->setup));
    in->footprint = footprint_of(p);
    in->ncell = L.n;
    in->id = ctx->next_id++;
    ctx->inst[in->id] = in;
    *id = in->id;
    return DBA_OK;
}

dba_status dba_instance_destroy(dba_ctx* ctx, int32_t id) {
    if (!ctx) return fail(DBA_ERR_INVALID, "null ctx");
    Instance* in = find(ctx, id);
    if (!in) return fail(DBA_ERR_NOTFOUND, "unknown instance %d", id);
    (void)hipStreamSynchronize(ctx->stream);
    ctx->unsettled.erase(std::remove(ctx->unsettled.begin(), ctx->unsettled.end(), id), ctx->unsettled.end());
    invalidate_groups(ctx, id);
    free_instance(in);
    ctx->inst.erase(id);
    delete in;
    return DBA_OK;
}

dba_status dba_instance_info(dba_ctx* ctx, int32_t id, dba_info* out) {
    if (!ctx || !out) return fail(DBA_ERR_INVALID, "null argument");
    Instance* in = find(ctx, id);
    if (!in) return fail(DBA_ERR_NOTFOUND, "unknown instance %d", id);
    WAIT_STREAM(ctx);
    double scal[16];
    int64_t ctr[4];
    HIP_TRY(hipMemcpy(scal, in->h.scal, sizeof(scal), hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(ctr, in->h.ctr, sizeof(ctr), hipMemcpyDeviceToHost));
    out->steps_done = ctr[0];
    out->field_updates = ctr[1];
    out->cell_updates = ctr[1] / std::max(1, in->h.nsets);
    out->ntiles = in->h.nt;
    out->ntiles_x = in->h.ntx;
    out->ntiles_y = in->h.nty;
    out->ntiles_z = in->h.ntz;
    out->sim_time = scal[2];
    out->last_dt = scal[3];
    out->cons_offset = scal[8];
    out->footprint_bytes = in->footprint;
    out->single_launch = ctx->single_launch != 0 && single_launch_params(in->p, in->h.nt) ? 1 : 0;
    out->reserved = 0;
    return DBA_OK;
}

dba_status dba_upload(dba_ctx* ctx, int32_t id, int32_t field, const double* host, size_t n) {
    if (!ctx || !host) return fail(DBA_ERR_INVALID, "null argument");
    Instance* in = find(ctx, id);
    if (!in) return fail(DBA_ERR_NOTFOUND, "unknown instance %d", id);
    if (field < 0 || field >= in->h.nfields) return fail(DBA_ERR_INVALID, "field %d invalid", field);
    if ((int64_t)n != in->ncell) return fail(DBA_ERR_INVALID, "n=%zu, expected %lld", n, (long long)in->ncell);
    // An instance that was never stepped is touched by no queued kernel, so its
    // upload overlaps the steps of other instances; otherwise it is ordered
    // after them on the compute stream.
    hipStream_t s = in->stepped ? ctx->stream : ctx->setup;
    DBA_TRY(settle(ctx, id));
    HIP_TRY(hipMemcpyAsync(in->h.buf[0][field], host, n * sizeof(double), hipMemcpyHostToDevice, s));
    HIP_TRY(hipMemcpyAsync(in->h.buf[1][field], in->h.buf[0][field], n * sizeof(double), hipMemcpyDeviceToDevice, s));
    if (in->h.ncons > 0) {
        hipLaunchKernelGGL(reset_epochs_kernel, dim3(64), dim3(256), 0, s, in->d_self, 0);
        LAUNCH_CHECK();
    }
    if (in->p.model == DBA_MODEL_KH) in->needs_prime = true;
    HIP_TRY(hipStreamSynchronize(s));
    return DBA_OK;
}

dba_status dba_download(dba_ctx* ctx, int32_t id, int32_t field, double* host, size_t n) {
    if (!ctx || !host) return fail(DBA_ERR_INVALID, "null argument");
    Instance* in = find(ctx, id);
    if (!in) return fail(DBA_ERR_NOTFOUND, "unknown instance %d", id);
    if (field < 0 || field >= in->h.nfields) return fail(DBA_ERR_INVALID, "field %d invalid", field);
    if ((int64_t)n != in->ncell) return fail(DBA_ERR_INVALID, "n=%zu, expected %lld", n, (long long)in->ncell);
    dba_status st = ensure_staging(ctx, n);
    if (st != DBA_OK) return st;
    unsigned blocks = (unsigned)std::min<int64_t>(4096, (in->ncell + 255) / 256);
    hipLaunchKernelGGL(materialize_kernel, dim3(blocks), dim3(256), 0, ctx->stream, in->d_self, 0, field,
                       ctx->staging);
    LAUNCH_CHECK();
    HIP_TRY(hipMemcpyAsync(host, ctx->staging, n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    WAIT_READ(ctx, dba_download(ctx, id, field, host, n));
    return DBA_OK;
}

dba_status dba_step(dba_ctx* ctx, const int32_t* ids, int32_t n_ids, int32_t n_steps) {
    if (!ctx) return fail(DBA_ERR_INVALID, "null ctx");
    if (n_steps < 0) return fail(DBA_ERR_INVALID, "n_steps < 0");
    std::vector<Group*> gs;
    dba_status st = prepare_groups(ctx, ids, n_ids, &gs);
    if (st != DBA_OK) return st;
    bool taken = false;
    if (gs.size() == 1) st = enqueue_resident(ctx, gs[0], n_steps, &taken);
    if (st != DBA_OK || taken) return st;
    DBA_TRY(settle_groups(ctx, ids, n_ids, &gs));
    return enqueue_steps(ctx, gs, n_steps, ctx->timing);
}

dba_status dba_step_graph(dba_ctx* ctx, const int32_t* ids, int32_t n_ids, int32_t n_steps, int32_t chunk) {
    if (!ctx) return fail(DBA_ERR_INVALID, "null ctx");
    if (n_steps < 0 || chunk < 1) return fail(DBA_ERR_INVALID, "n_steps < 0 or chunk < 1");
    std::vector<Group*> gs;
    dba_status st = prepare_groups(ctx, ids, n_ids, &gs);
    if (st != DBA_OK) return st;
    bool taken = false;
    if (gs.size() == 1) st = enqueue_resident(ctx, gs[0], n_steps, &taken);
    if (st != DBA_OK || taken) return st;
    DBA_TRY(settle_groups(ctx, ids, n_ids, &gs));
    int reps = n_steps / chunk, rem = n_steps % chunk;
    if (reps > 0) {
        GraphKey key{std::vector<int>(ids, ids + n_ids), chunk, ctx->single_launch};
        auto it = ctx->graphs.find(key);
        hipGraphExec_t exec = nullptr;
        if (it == ctx->graphs.end()) {
            evict_graphs(ctx);
            hipGraph_t graph = nullptr;
            HIP_TRY(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeRelaxed));
            dba_status est = enqueue_steps(ctx, gs, chunk, false);
            hipError_t e = hipStreamEndCapture(ctx->stream, &graph);
            if (est != DBA_OK) return est;
            if (e != hipSuccess) return fail(DBA_ERR_HIP, "hipStreamEndCapture: %s", hipGetErrorString(e));
            HIP_TRY(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
            (void)hipGraphDestroy(graph);
            ctx->graphs[key] = CachedGraph{exec, ctx->clock};
        } else {
            it->second.last_use = ctx->clock;
            exec = it->second.exec;
        }
        for (int r = 0; r < reps; r++) HIP_TRY(hipGraphLaunch(exec, ctx->stream));
    }
    if (rem > 0) return enqueue_steps(ctx, gs, rem, false);
    return DBA_OK;
}

dba_status dba_set_single_launch(dba_ctx* ctx, int32_t mode) {
    if (!ctx) return fail(DBA_ERR_INVALID, "null ctx");
    if (mode < 0 || mode > 2) return fail(DBA_ERR_INVALID, "single-launch mode must be 0, 1 or 2 (got %d)", mode);
    // captured graphs are cached per mode, so switching keeps them
    ctx->single_launch = mode;
    return DBA_OK;
}

dba_status dba_set_resident(dba_ctx* ctx, int32_t enable) {
    if (!ctx) return fail(DBA_ERR_INVALID, "null ctx");
    ctx->resident = enable != 0;
    return DBA_OK;
}

dba_status dba_set_resident_wait(dba_ctx* ctx, int32_t polls) {
    if (!ctx) return fail(DBA_ERR_INVALID, "null ctx");
    if (polls < 0) return fail(DBA_ERR_INVALID, "polls < 0");
    ctx->wait_polls = polls ? polls : kWaitPolls;
    return DBA_OK;
}

dba_status dba_resident_calls(dba_ctx* ctx, int64_t* taken) {
    if (!ctx || !taken) return fail(DBA_ERR_INVALID, "null argument");
    *taken = ctx->resident_calls;
    return DBA_OK;
}

dba_status dba_resident_redone(dba_ctx* ctx, int64_t* steps) {
    if (!ctx || !steps) return fail(DBA_ERR_INVALID, "null argument");
    *steps = ctx->resident_redone;
    return DBA_OK;
}

dba_status dba_sync(dba_ctx* ctx) {
    if (!ctx) return fail(DBA_ERR_INVALID, "null ctx");
    WAIT_STREAM(ctx);
    return DBA_OK;
}

dba_status dba_active_tiles(dba_ctx* ctx, int32_t id, int32_t set, int32_t* count, uint8_t* mask) {
    if (!ctx || !count) return fail(DBA_ERR_INVALID, "null argument");
    Instance* in = find(ctx, id);
    if (!in) return fail(DBA_ERR_NOTFOUND, "unknown instance %d", id);
    if (set < 0 || set >= in->h.nsets) return fail(DBA_ERR_INVALID, "set %d invalid", set);
    WAIT_STREAM(ctx);
    int nt = in->h.nt;
    std::vector<uint64_t> w((size_t)in->h.nwords);
    HIP_TRY(hipMemcpy(w.data(), in->h.a_cur[set], sizeof(uint64_t) * w.size(), hipMemcpyDeviceToHost));
    int c = 0;
    for (int t = 0; t < nt; t++) {
        int b = in->p.mode == DBA_MODE_REGULAR ? 1 : (int)((w[t >> 6] >> (t & 63)) & 1ull);
        c += b;
        if (mask) mask[t] = (uint8_t)b;
    }
    *count = c;
    return DBA_OK;
}

dba_status dba_worklist(dba_ctx* ctx, int32_t id, int32_t* tiles, int32_t cap, int32_t* count) {
    if (!ctx || !count) return fail(DBA_ERR_INVALID, "null argument");
    Instance* in = find(ctx, id);
    if (!in) return fail(DBA_ERR_NOTFOUND, "unknown instance %d", id);
    // compact the instance's current awake set (the list the next step runs)
    DBA_TRY(settle(ctx, id));
    std::vector<Group*> gs;
    dba_status st = prepare_groups(ctx, &id, 1, &gs);
    if (st != DBA_OK) return st;
    WAIT_STREAM(ctx);
    int64_t ctr[4];
    HIP_TRY(hipMemcpy(ctr, in->h.ctr, sizeof(ctr), hipMemcpyDeviceToHost));
    *count = (int32_t)ctr[2];
    if (tiles && cap > 0) {
        int n = (int)std::min<int64_t>(cap, ctr[2]);
        if (n > 0) HIP_TRY(hipMemcpy(tiles, in->h.seg, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
    }
    return DBA_OK;
}

dba_status dba_active_history(dba_ctx* ctx, int32_t id, int32_t* counts, int32_t max_steps, int32_t* n_steps) {
    if (!ctx || !n_steps) return fail(DBA_ERR_INVALID, "null argument");
    Instance* in = find(ctx, id);
    if (!in) return fail(DBA_ERR_NOTFOUND, "unknown instance %d", id);
    WAIT_STREAM(ctx);
    int64_t ctr[4];
    HIP_TRY(hipMemcpy(ctr, in->h.ctr, sizeof(ctr), hipMemcpyDeviceToHost));
    int n = (int)std::min<int64_t>(std::min<int64_t>(ctr[0], in->h.hist_cap), max_steps);
    if (counts && n > 0) HIP_TRY(hipMemcpy(counts, in->h.hist, sizeof(int32_t) * 2 * n, hipMemcpyDeviceToHost));
    *n_steps = n;
    return DBA_OK;
}

dba_status dba_timing_enable(dba_ctx* ctx, int32_t enable) {
    if (!ctx) return fail(DBA_ERR_INVALID, "null ctx");
    WAIT_STREAM(ctx);
    ctx->ev_pool.insert(ctx->ev_pool.end(), ctx->ev_used.begin(), ctx->ev_used.end());
    ctx->ev_used.clear();
    ctx->ev_step.clear();
    ctx->ev_fin.clear();
    ctx->timing = enable != 0;
    return DBA_OK;
}

dba_status dba_timing_query(dba_ctx* ctx, double* step_ms, int64_t* step_n, double* fin_ms, int64_t* fin_n) {
    if (!ctx) return fail(DBA_ERR_INVALID, "null ctx");
    WAIT_STREAM(ctx);
    double a = 0.0, b = 0.0;
    for (auto& e : ctx->ev_step) {
        float ms = 0.f;
        HIP_TRY(hipEventElapsedTime(&ms, e.first, e.second));
        a += ms;
    }
    for (auto& e : ctx->ev_fin) {
        float ms = 0.f;
        HIP_TRY(hipEventElapsedTime(&ms, e.first, e.second));
        b += ms;
    }
    if (step_ms) *step_ms = a;
    if (step_n) *step_n = (int64_t)ctx->ev_step.size();
    if (fin_ms) *fin_ms = b;
    if (fin_n) *fin_n = (int64_t)ctx->ev_fin.size();
    return DBA_OK;
}

dba_status dba_marker(dba_ctx* ctx, int32_t slot) {
    if (!ctx || slot < 0 || slot >= 8) return fail(DBA_ERR_INVALID, "bad marker slot");
    HIP_TRY(hipEventRecord(ctx->markers[slot], ctx->stream));
    return DBA_OK;
}

dba_status dba_marker_elapsed(dba_ctx* ctx, int32_t a, int32_t b, double* ms) {
    if (!ctx || !ms || a < 0 || a >= 8 || b < 0 || b >= 8) return fail(DBA_ERR_INVALID, "bad marker slot");
    HIP_TRY(hipEventSynchronize(ctx->markers[b]));
    float f = 0.f;
    HIP_TRY(hipEventElapsedTime(&f, ctx->markers[a], ctx->markers[b]));
    *ms = f;
    return DBA_OK;
}

dba_status dba_check_finite(dba_ctx* ctx, int32_t id) {
    if (!ctx) return fail(DBA_ERR_INVALID, "null ctx");
    Instance* in = find(ctx, id);
    if (!in) return fail(DBA_ERR_NOTFOUND, "unknown instance %d", id);
    HIP_TRY(hipMemsetAsync(ctx->d_flag, 0, sizeof(int), ctx->stream));
    unsigned blocks = (unsigned)std::min<int64_t>(2048, (in->ncell + 255) / 256);
    hipLaunchKernelGGL(finite_kernel, dim3(blocks), dim3(256), 0, ctx->stream, in->d_self, 0, ctx->d_flag);
    LAUNCH_CHECK();
    int bad = 0;
    HIP_TRY(hipMemcpyAsync(&bad, ctx->d_flag, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    WAIT_READ(ctx, dba_check_finite(ctx, id));
    if (bad) return fail(DBA_ERR_NUMERIC, "instance %d holds non-finite values", id);
    return DBA_OK;
}

dba_status dba_field_sum(dba_ctx* ctx, int32_t id, int32_t field, double* sum) {
    if (!ctx || !sum) return fail(DBA_ERR_INVALID, "null argument");
    Instance* in = find(ctx, id);
    if (!in) return fail(DBA_ERR_NOTFOUND, "unknown instance %d", id);
    if (field < 0 || field >= in->h.nfields) return fail(DBA_ERR_INVALID, "field %d invalid", field);
    double* part = ctx->d_diag;
    double* res = ctx->d_diag + 3 * kDiagBlocks;
    hipLaunchKernelGGL(field_sum_kernel, dim3(kDiagBlocks), dim3(kDiagNT), 0, ctx->stream, in->d_self, 0, field,
                       part);
    LAUNCH_CHECK();
    hipLaunchKernelGGL(reduce_parts_kernel, dim3(1), dim3(64), 0, ctx->stream, part, 1, res);
    LAUNCH_CHECK();
    HIP_TRY(hipMemcpyAsync(sum, res, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    WAIT_READ(ctx, dba_field_sum(ctx, id, field, sum));
    return DBA_OK;
}

dba_status dba_growth_front(dba_ctx* ctx, int32_t id, const int32_t* xs, int32_t n, double* front) {
    if (!ctx || !xs || !front) return fail(DBA_ERR_INVALID, "null argument");
    Instance* in = find(ctx, id);
    if (!in) return fail(DBA_ERR_NOTFOUND, "unknown instance %d", id);
    if (in->p.model != DBA_MODEL_DENDRITE_K93 && in->p.model != DBA_MODEL_DENDRITE_K94)
        return fail(DBA_ERR_INVALID, "growth front needs a dendrite instance");
    if (n < 0 || n > kMaxFrontCols) return fail(DBA_ERR_INVALID, "n must be in [0, %d]", kMaxFrontCols);
    for (int k = 0; k < n; k++)
        if (xs[k] < 0 || xs[k] >= in->p.nx) return fail(DBA_ERR_INVALID, "column %d outside the grid", xs[k]);
    if (n == 0) return DBA_OK;
    // synchronous so the host array may be reused at once; ordered after queued steps
    HIP_TRY(hipMemcpyAsync(ctx->d_cols, xs, sizeof(int32_t) * n, hipMemcpyHostToDevice, ctx->stream));
    double* res = ctx->d_diag + 3 * kDiagBlocks;
    hipLaunchKernelGGL(growth_front_kernel, dim3(1), dim3(kMaxFrontCols), 0, ctx->stream, in->d_self, 0,
                       ctx->d_cols, n, res);
    LAUNCH_CHECK();
    HIP_TRY(hipMemcpyAsync(front, res, sizeof(double) * n, hipMemcpyDeviceToHost, ctx->stream));
    WAIT_READ(ctx, dba_growth_front(ctx, id, xs, n, front));
    return DBA_OK;
}

dba_status dba_droplets(dba_ctx* ctx, int32_t id, int32_t field, double* avg, int64_t* volume,
                        int64_t* n_droplets, int64_t* sizes, int64_t cap) {
    if (!ctx || !avg || !volume || !n_droplets) return fail(DBA_ERR_INVALID, "null argument");
    if (cap < 0 || (cap > 0 && !sizes)) return fail(DBA_ERR_INVALID, "sizes must hold cap >= 0 entries");
    Instance* in = find(ctx, id);
    if (!in) return fail(DBA_ERR_NOTFOUND, "unknown instance %d", id);
    if (field < 0 || field >= in->h.nfields) return fail(DBA_ERR_INVALID, "field %d invalid", field);
    const int64_t n = (int64_t)in->p.nx * in->p.ny * in->p.nz;
    if (n >= INT32_MAX) return fail(DBA_ERR_INVALID, "droplet analysis supports grids below 2^31 cells");
    CcScratch sc;
    uint8_t* cls;
    int32_t *parent, *size, *key;
    double *part, *d_avg;
    int64_t *vpart, *counters;
    if (sc.get(&cls, n) != hipSuccess || sc.get(&parent, n) != hipSuccess || sc.get(&size, n) != hipSuccess ||
        sc.get(&key, n) != hipSuccess || sc.get(&part, 2 * kCcBlocks) != hipSuccess || sc.get(&d_avg, 1) != hipSuccess ||
        sc.get(&vpart, kCcBlocks) != hipSuccess || sc.get(&counters, 2) != hipSuccess)
        return fail(DBA_ERR_NOMEM, "droplet analysis: no device memory for %lld cells", (long long)n);
    hipStream_t st = ctx->stream;
    const dim3 g(kCcBlocks), b(kCcNT);
    hipLaunchKernelGGL(cc_minmax_kernel, g, b, 0, st, in->d_self, 0, field, part);
    hipLaunchKernelGGL(cc_threshold_kernel, dim3(1), dim3(64), 0, st, part, d_avg);
    hipLaunchKernelGGL(cc_init_kernel, g, b, 0, st, in->d_self, 0, field, d_avg, cls, parent, size, key);
    hipLaunchKernelGGL(cc_union_kernel, g, b, 0, st, cls, parent, in->p.nx, in->p.ny, in->p.nz);
    hipLaunchKernelGGL(cc_count_kernel, g, b, 0, st, cls, parent, size, key, n, vpart);
    HIP_TRY(hipMemsetAsync(counters, 0, 2 * sizeof(int64_t), st));
    hipLaunchKernelGGL(cc_collect_kernel, g, b, 0, st, size, key, n, vpart, counters, (int64_t*)nullptr,
                       (int64_t)0);
    LAUNCH_CHECK();
    int64_t cnt[2];
    HIP_TRY(hipMemcpyAsync(cnt, counters, sizeof(cnt), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipMemcpyAsync(avg, d_avg, sizeof(double), hipMemcpyDeviceToHost, st));
    WAIT_READ(ctx, dba_droplets(ctx, id, field, avg, volume, n_droplets, sizes, cap));
    *n_droplets = cnt[0];
    *volume = cnt[1];
    if (cap == 0 || cnt[0] == 0) return DBA_OK;
    // second pass with room for every droplet, then the reference's order:
    // droplets by their first seed in index order
    int64_t* pairs;
    if (sc.get(&pairs, 2 * cnt[0]) != hipSuccess) return fail(DBA_ERR_NOMEM, "droplet analysis: no device memory");
    HIP_TRY(hipMemsetAsync(counters, 0, sizeof(int64_t), st));
    hipLaunchKernelGGL(cc_collect_kernel, g, b, 0, st, size, key, n, vpart, counters, pairs, cnt[0]);
    LAUNCH_CHECK();
    std::vector<int64_t> h((size_t)(2 * cnt[0]));
    HIP_TRY(hipMemcpyAsync(h.data(), pairs, sizeof(int64_t) * h.size(), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    std::vector<std::pair<int64_t, int64_t>> v((size_t)cnt[0]);
    for (int64_t k = 0; k < cnt[0]; k++) v[(size_t)k] = {h[(size_t)(2 * k)], h[(size_t)(2 * k + 1)]};
    std::sort(v.begin(), v.end());
    for (int64_t k = 0; k < cnt[0] && k < cap; k++) sizes[k] = v[(size_t)k].second;
    return DBA_OK;
}

dba_status dba_droplets_noalloc(dba_ctx* ctx, int32_t id, int32_t field, double* avg, int64_t* volume,
                                int64_t* n_droplets, int64_t* sizes, int64_t cap) {
    if (!ctx || !avg || !volume || !n_droplets) return fail(DBA_ERR_INVALID, "null argument");
    if (cap < 0 || (cap > 0 && !sizes)) return fail(DBA_ERR_INVALID, "sizes must hold cap >= 0 entries");
    Instance* in = find(ctx, id);
    if (!in) return fail(DBA_ERR_NOTFOUND, "unknown instance %d", id);
    if (field < 0 || field >= in->h.nfields) return fail(DBA_ERR_INVALID, "field %d invalid", field);
    const int64_t n = (int64_t)in->p.nx * in->p.ny * in->p.nz;
    if (n > kScratchMaxCells)
        return fail(DBA_ERR_INVALID,
                    "dba_droplets_noalloc: %lld cells exceed the static scratch of %lld cells; use dba_droplets",
                    (long long)n, (long long)kScratchMaxCells);
    // carve the scratch: every region 256-byte aligned, at most kScratchBytes in all
    unsigned char* q = ctx->scratch;
    auto take = [&q](size_t bytes) {
        unsigned char* r = q;
        q += (bytes + 255) & ~(size_t)255;
        return r;
    };
    uint8_t* cls = take((size_t)n);
    int32_t* parent = (int32_t*)take(4 * (size_t)n);
    int32_t* size = (int32_t*)take(4 * (size_t)n);
    int32_t* key = (int32_t*)take(4 * (size_t)n);
    double* part = (double*)take(sizeof(double) * 2 * kCcBlocks);
    double* d_avg = (double*)take(sizeof(double));
    int64_t* vpart = (int64_t*)take(sizeof(int64_t) * kCcBlocks);
    int64_t* counters = (int64_t*)take(sizeof(int64_t) * 2);
    int32_t* bcount = (int32_t*)take(sizeof(int32_t) * kCcBlocks);
    if ((size_t)(q - ctx->scratch) > kScratchBytes)
        return fail(DBA_ERR_INVALID, "dba_droplets_noalloc: scratch layout exceeds its array");
    hipStream_t st = ctx->stream;
    const dim3 g(kCcBlocks), b(kCcNT);
    hipLaunchKernelGGL(cc_minmax_kernel, g, b, 0, st, in->d_self, 0, field, part);
    hipLaunchKernelGGL(cc_threshold_kernel, dim3(1), dim3(64), 0, st, part, d_avg);
    hipLaunchKernelGGL(cc_init_kernel, g, b, 0, st, in->d_self, 0, field, d_avg, cls, parent, size, key);
    hipLaunchKernelGGL(cc_union_kernel, g, b, 0, st, cls, parent, in->p.nx, in->p.ny, in->p.nz);
    hipLaunchKernelGGL(cc_count_kernel, g, b, 0, st, cls, parent, size, key, n, vpart);
    // the forest is done with: parent[] becomes first[]
    hipLaunchKernelGGL(cc_fill_kernel, g, b, 0, st, parent, n, 0, counters);
    hipLaunchKernelGGL(cc_mark_kernel, g, b, 0, st, size, key, n, vpart, parent, counters);
    LAUNCH_CHECK();
    int64_t cnt[2];
    HIP_TRY(hipMemcpyAsync(cnt, counters, sizeof(cnt), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipMemcpyAsync(avg, d_avg, sizeof(double), hipMemcpyDeviceToHost, st));
    WAIT_READ(ctx, dba_droplets_noalloc(ctx, id, field, avg, volume, n_droplets, sizes, cap));
    *n_droplets = cnt[0];
    *volume = cnt[1];
    if (cap == 0 || cnt[0] == 0) return DBA_OK;
    // the droplets in the order of their first seeds, compacted into size[]
    const int64_t chunk = ((n + kCcBlocks - 1) / kCcBlocks + kCcNT - 1) / kCcNT * kCcNT;
    const int64_t k = std::min<int64_t>(cap, cnt[0]);
    hipLaunchKernelGGL(cc_order_count_kernel, g, b, 0, st, parent, n, chunk, bcount);
    hipLaunchKernelGGL(cc_order_write_kernel, g, b, 0, st, parent, n, chunk, bcount, size, k);
    LAUNCH_CHECK();
    // k int32 sizes into the front of the caller's int64 array, then widened in
    // place from the back (entry j is read before slot j's bytes are written)
    int32_t* narrow = (int32_t*)sizes;
    HIP_TRY(hipMemcpyAsync(narrow, size, sizeof(int32_t) * (size_t)k, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    for (int64_t j = k - 1; j >= 0; j--) sizes[j] = (int64_t)narrow[j];
    return DBA_OK;
}

dba_status dba_kh_vy_mode(dba_ctx* ctx, int32_t id, double* amplitude) {
    if (!ctx || !amplitude) return fail(DBA_ERR_INVALID, "null argument");
    Instance* in = find(ctx, id);
    if (!in) return fail(DBA_ERR_NOTFOUND, "unknown instance %d", id);
    if (in->p.model != DBA_MODEL_KH) return fail(DBA_ERR_INVALID, "vy mode needs a KH instance");
    double* part = ctx->d_diag;
    double* res = ctx->d_diag + 3 * kDiagBlocks;
    hipLaunchKernelGGL(vy_mode_kernel, dim3(kDiagBlocks), dim3(kDiagNT), 0, ctx->stream, in->d_self, 0, part);
    LAUNCH_CHECK();
    hipLaunchKernelGGL(reduce_parts_kernel, dim3(1), dim3(64), 0, ctx->stream, part, 3, res);
    LAUNCH_CHECK();
    double s[3];
    HIP_TRY(hipMemcpyAsync(s, res, sizeof(s), hipMemcpyDeviceToHost, ctx->stream));
    WAIT_STREAM(ctx);
    *amplitude = 2.0 * std::sqrt(s[0] * s[0] / (s[2] * s[2]) + s[1] * s[1] / (s[2] * s[2]));
    return DBA_OK;
}

}  // extern "C"
