// k_resident.h - many DBA steps of one instance in one cooperative launch, the
// fields in LDS from the first step to the last.
//
// A step of a grid that fits the chip is bound by latency, not by bytes or
// arithmetic: with one launch per step a 1024^2 Cahn-Hilliard step takes 7 us, of
// which a copy of the grid would take 3 and the arithmetic 2; the rest is the gap
// between launches, the tables every workgroup builds first and the trip of every
// cell through the caches. Here each workgroup owns a region of gx x gy tiles for
// the whole call, keeps its cells in LDS, and per step exchanges only the two-cell
// frame its neighbours read.
//
// Exchange: every published value travels as two 8-byte words, each holding half
// of the double and the step's sequence number, written and read with relaxed
// atomics of agent scope (they bypass the per-XCD caches). A word is valid when its
// number is the expected one, so there is no flag to wait for after the data and
// no fence. Two generations (step parity) suffice: a tile publishes generation
// s + 2 only after step s + 1, for which it has received every neighbour's word of
// step s, and those were sent after the neighbour had read generation s.
//
// Progress: the launch is cooperative and its size is checked against the chip, so all
// workgroups are resident unless something else holds compute units (another process);
// a workgroup waits only for words of the step before, which their owners send without
// waiting for anything of this step, so by induction over the steps every wait ends.
// Each wait is bounded all the same: a workgroup past the bound gives the launch up and
// ends; those that wait for its words run out a few steps later, those that only get a
// place on the chip then see it as they start, and the host has the steps made on
// another path. So a launch that is given up leaves the instance as it was. What it
// stores before its end only counts once the canonicalising kernel takes it over (the
// cells go to the buffers that are not current); what replaces state in place (the
// stored potential rings of CH) waits until every workgroup has made all its steps
// (resident_all_done).
#pragma once
#include "common.h"
#include "k_ch.h"
#include "k_finalize.h"

namespace dba {

// State of the context's resident launches, in front of the exchange's frames (a pointer
// of its own would be one more to keep in registers through the steps). A launch that
// starts with kResGivenUp makes no steps: the host has not taken notice of the one before
// it yet.
constexpr uint32_t kResRunning = 0, kResGivenUp = 1, kResDone = 2;
struct ResHead {
    uint32_t state, done;  // done: workgroups that have made all their steps
    int* stuck;            // host memory: a launch was given up
    uint64_t pad[14];      // a cache line of its own
};

struct Exchange {
    uint64_t* frame;   // [parity][region][slot][2 words per field]
    uint64_t* flag;    // [parity][tile]: sequence number << 32 | detector bits
    int polls;         // polls after which a wait is given up
    uint32_t base;     // sequence number of the launch's first step
    int slots;         // frame slots of a whole region
    __device__ __forceinline__ ResHead* head() const { return (ResHead*)frame - 1; }
};

__device__ __forceinline__ void xput(uint64_t* p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t xget(const uint64_t* p) {
    return __hip_atomic_load((uint64_t*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void put_double(uint64_t* p, double v, uint32_t seq) {
    const uint64_t b = (uint64_t)__double_as_longlong(v), s = (uint64_t)seq << 32;
    xput(p, s | (uint32_t)b);
    xput(p + 1, s | (uint32_t)(b >> 32));
}

// Bound of a wait, if the caller sets none: about a second of polls (each is a trip to
// memory). Other work of the process may hold compute units that a workgroup of the
// launch still needs, and a launch given up costs that second once: the context then
// keeps to the other paths.
constexpr int kWaitPolls = 1 << 20;

__device__ __forceinline__ uint32_t resident_state(const Exchange& X) {
    return __hip_atomic_load(&X.head()->state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ bool resident_end(const Exchange& X, uint32_t how) {
    uint32_t s = kResRunning;
    return __hip_atomic_compare_exchange_strong(&X.head()->state, &s, how, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
}

// Gives the launch up, unless it is done (one thread).
__device__ __forceinline__ void resident_give_up(const Exchange& X) {
    if (resident_end(X, kResGivenUp)) __hip_atomic_store(X.head()->stuck, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// One thread of a workgroup that has made all its steps: true once all workgroups have,
// false if the launch was given up instead. A workgroup that has nothing to hold back
// does not wait (the wait cost a 20-step call 3 us: a trip to memory and the last one's lag).
__device__ __forceinline__ bool resident_all_done(const Exchange& X, bool wait) {
    __hip_atomic_fetch_add(&X.head()->done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (!wait) return true;
    for (int k = 0;; k++) {
        const uint32_t s = resident_state(X);
        if (s != kResRunning) return s == kResDone;
        if (__hip_atomic_load(&X.head()->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x)
            resident_end(X, kResDone);
        else if (k >= X.polls)
            resident_give_up(X);
    }
}

// A word of another workgroup. Past the bound only *gone is set: what giving up takes is
// kept out of the loops, where its registers cost 2% of a step.
__device__ __forceinline__ double wait_double(const uint64_t* p, uint32_t seq, const Exchange& X, int* gone) {
    uint64_t a, b;
    for (int k = 0;; k++) {
        a = xget(p);
        b = xget(p + 1);
        if ((uint32_t)(a >> 32) == seq && (uint32_t)(b >> 32) == seq) break;
        if (k >= X.polls) {
            *gone = 1;
            break;
        }
    }
    return __longlong_as_double((long long)((uint64_t)(uint32_t)b << 32 | (uint32_t)a));
}

__device__ __forceinline__ int wait_flag(const uint64_t* p, uint32_t seq, const Exchange& X, int* gone) {
    uint64_t a;
    for (int k = 0;; k++) {
        a = xget(p);
        if ((uint32_t)(a >> 32) == seq) break;
        if (k >= X.polls) {
            *gone = 1;
            break;
        }
    }
    return (int)(a & 3ull);
}

// The published cells of a w x h region: two cells deep on each side, every cell
// one slot (rows first, so the cells of a region two or three cells thick have one).
__host__ __device__ __forceinline__ int frame_slots(int w, int h) { return 4 * w + 4 * h; }  // at most

__device__ __forceinline__ int frame_slot(int lx, int ly, int w, int h) {
    if (ly < 2) return ly * w + lx;
    if (ly >= h - 2) return 2 * w + (ly - (h - 2)) * w + lx;
    if (lx < 2) return 4 * w + (ly - 2) * 2 + lx;
    if (lx >= w - 2) return 4 * w + 2 * (h - 4) + (ly - 2) * 2 + (lx - (w - 2));
    return -1;
}

// cell k of the ring of thickness T around a w x h region (coordinates from -T):
// the rows below, the rows above, then the columns
template <int T>
__device__ __forceinline__ void outer_cell(int k, int w, int h, int* x, int* y) {
    const int W = w + 2 * T;
    if (k < 2 * T * W) {
        const int r = k / W;
        *y = r < T ? r - T : h + r - T;
        *x = k - r * W - T;
    } else {
        const int q = k - 2 * T * W, c = q % (2 * T);
        *y = q / (2 * T);
        *x = c < T ? c - T : w + c - T;
    }
}

constexpr int kResMaxTiles = 16;  // tiles of a region, at most (with their surroundings two deep: 64, one ballot)

struct ResTile {
    int t, x, y, w, h, par, runs, last;  // tile, window position, extent, buffer, steps run, bit of the last of them
    int pos;                             // position among the awake bits
};

// LDS bytes of a region of w x h cells.
constexpr size_t ch_resident_bytes(int w, int h) {
    return sizeof(double) * ((size_t)(w + 4) * (h + 4) + (size_t)(w + 2) * (h + 2));
}

// Threads a region of w x h cells needs at least: one for each cell of its halo (and
// of its mu ring and edge), whose place and owner that thread keeps in registers.
constexpr int ch_resident_threads(int w, int h) { return 4 * (w + h) + 16; }

// A workgroup's region: gx x gy tiles of TB x TB (fewer at the grid's end), its cells
// from (x0, y0), and the positions of its tiles and the two tiles around it on every
// side: tile (i, j) of the region at (i + 2) + (j + 2) PW.
template <int TB>
struct Region {
    int nx, ny, ntx, nty, bcx, bcy, gx, gy, nrx, rgn, ti0, tj0, kx, ky, nk, x0, y0, w, h, PW;

    __device__ __forceinline__ Region(CInst& I, int gx_, int gy_)
        : nx(I.nx), ny(I.ny), ntx(I.ntx), nty(I.nty), bcx(I.bc_x), bcy(I.bc_y), gx(gx_), gy(gy_),
          nrx((I.ntx + gx_ - 1) / gx_), rgn(blockIdx.x) {
        ti0 = rgn % nrx * gx;
        tj0 = rgn / nrx * gy;
        kx = min(gx, ntx - ti0);
        ky = min(gy, nty - tj0);
        nk = kx * ky;
        x0 = ti0 * TB;
        y0 = tj0 * TB;
        w = min(kx * TB, nx - x0);
        h = min(ky * TB, ny - y0);
        PW = kx + 4;
    }
    // the tile at position p, or -1 outside a closed boundary or past the positions
    __device__ __forceinline__ int near(int p) const {
        if (p >= PW * (ky + 4)) return -1;
        int i = ti0 + p % PW - 2, j = tj0 + p / PW - 2;
        if (bcx == 0) i = ((i % ntx) + ntx) % ntx;
        if (bcy == 0) j = ((j % nty) + nty) % nty;
        return i >= 0 && i < ntx && j >= 0 && j < nty ? i + j * ntx : -1;
    }
    // the region's tile (i + j kx) at position p, or -1
    __device__ __forceinline__ int inside(int p) const {
        const int i = p % PW - 2, j = p / PW - 2;
        return i >= 0 && i < kx && j >= 0 && j < ky ? i + j * kx : -1;
    }
    // position of the tile that holds the mapped cell of (x, y), a cell outside the
    // region: mirrored cells belong to the region's own tiles
    __device__ __forceinline__ int pos_of(int x, int y) const {
        const int gxx = x0 + x, gyy = y0 + y;
        int i, j;
        if (bcx != 0 && (gxx < 0 || gxx >= nx)) i = map_index(gxx, nx, bcx) / TB - ti0;
        else i = x < 0 ? -1 : (x >= w ? kx : x / TB);
        if (bcy != 0 && (gyy < 0 || gyy >= ny)) j = map_index(gyy, ny, bcy) / TB - tj0;
        else j = y < 0 ? -1 : (y >= h ? ky : y / TB);
        return (i + 2) + (j + 2) * PW;
    }
    // mapped cell of (x, y): its tile, and its slot among the frames of all regions
    __device__ __forceinline__ void source(int x, int y, int slots, int* mx, int* my, int* tile, int* slot) const {
        *mx = map_index(x0 + x, nx, bcx);
        *my = map_index(y0 + y, ny, bcy);
        const int oi = *mx / TB, oj = *my / TB, ox = oi / gx, oy = oj / gy, bx = ox * gx * TB, by = oy * gy * TB;
        *tile = oi + oj * ntx;
        *slot = (ox + oy * nrx) * slots +
                frame_slot(*mx - bx, *my - by, min(gx * TB, nx - bx), min(gy * TB, ny - by));
    }
    // awake positions of a step from the detector bits of the step before
    __device__ __forceinline__ uint64_t dilate(uint64_t m, uint64_t exist) const {
        return (m | m << 1 | m >> 1 | m << PW | m >> PW) & exist;  // (rows touch only past the positions in use)
    }
};

// n steps of one CH instance (regular or DBA). The region's c (with a two-cell
// halo) and mu (with a one-cell ring) stay in LDS windows for the whole launch; per
// tile and step the arithmetic, its order and the detector are ch_tile's, so results
// are bit-identical to the other paths. A sleeping tile's mu is what the window
// still holds from the last step it ran, and a sleeping outside tile's ring is what
// this region computed for it then (the same doubles from the same cells); only at
// the end of the launch do tiles that did not fire when they last ran store their
// ring. The canonicalising kernels follow, as after single-launch steps.
//
// A step: 1. mu of the tiles that fired in the step before (they run whatever their
// neighbours did), all but the region's edge, while the frames of the other regions
// are on their way; 2. the halo and the outside detector bits; 3. mu of tiles only a
// neighbour woke, of the edge and of the ring; 4. c' and the frame.
// NT threads work on a tile: R = TB TB / NT rows of one column each.
template <int TB, int NT, bool NINE>
__global__ __launch_bounds__(1024) void ch_resident_kernel(const Inst* __restrict__ insts, Exchange X, int n, int gx,
                                                           int gy) {
    constexpr int R = TB * TB / NT;
    extern __shared__ __align__(16) double lds[];
    __shared__ ResTile tiles[kResMaxTiles];
    __shared__ int fire[3][kResMaxTiles];  // detector bits of step s in fire[s % 3]
    __shared__ int gone[2];                // a wait of step s ran out: gone[s & 1]
    __shared__ uint64_t sact[2];           // awake tiles of step s: positions of the region and two tiles around it
    CInst& I = ((CInst*)insts)[0];
    const int tid = threadIdx.x, lane = tid & 63, nthr = blockDim.x;
    const Region<TB> G(I, gx, gy);
    const int nx = G.nx, ny = G.ny, ntx = G.ntx, ti0 = G.ti0, tj0 = G.tj0, kx = G.kx, nk = G.nk;
    const int x0 = G.x0, y0 = G.y0, w = G.w, h = G.h, PW = G.PW, rgn = G.rgn;
    const bool regular = I.mode == 0;
    const double kappa = I.kappa, eps = I.thresh_a, inv = NINE ? I.inv6dx2 : I.invdx2;
    const double dt = I.dt, mob = I.mobility, rg = I.react_gamma, cbar = I.cbar;
    gdouble* mu_store = I.aux[0];
    const int W2 = w + 4, W1 = w + 2;
    const int nh = W2 * (h + 4) - w * h, nr = W1 * (h + 2) - w * h, ne = 2 * w + 2 * h - 4;
    double* sc = lds;                         // c at (x, y): sc[x + 2 + (y + 2) W2]
    double* smu = sc + (size_t)W2 * (h + 4);  // mu at (x, y): smu[x + 1 + (y + 1) W1]
    const int64_t plane = (int64_t)gridDim.x * X.slots * 2;

    const int near = G.near(lane);  // the tile at this lane's position

    // ---- tables and the state the launch starts from
    if (tid < nk) {
        const int i = tid % kx, j = tid / kx;
        ResTile& T = tiles[tid];
        T.t = (ti0 + i) + (tj0 + j) * ntx;
        T.x = i * TB;
        T.y = j * TB;
        T.w = min(TB, w - T.x);
        T.h = min(TB, h - T.y);
        T.par = bit_of(I.par[0], T.t);
        T.runs = 0;
        T.last = 1;
        T.pos = (i + 2) + (j + 2) * PW;
        for (int q = 0; q < 3; q++) fire[q][tid] = 0;
    }
    if (tid < 64) {
        const int a = near >= 0 && (regular || bit_of(I.a_cur[0], near));
        const uint64_t m = __ballot(a);
        if (lane == 0) {
            sact[0] = m;
            sact[1] = 0ull;
            gone[0] = resident_state(X) == kResGivenUp;
            gone[1] = 0;
        }
    }
    for (int k = tid; k < w * h; k += nthr) {
        const int x = k % w, y = k / w, t = (ti0 + x / TB) + (tj0 + y / TB) * ntx;
        sc[(x + 2) + (y + 2) * W2] = I.buf[bit_of(I.par[0], t)][0][(x0 + x) + (int64_t)(y0 + y) * nx];
    }
    // this thread's cell of the halo: where it is published, the tile position of its owner, its place
    int hslot = 0, hpos = -1, hcell = 0;
    if (tid < nh) {
        int x, y;
        outer_cell<2>(tid, w, h, &x, &y);
        int mx, my, tile;
        G.source(x, y, X.slots, &mx, &my, &tile, &hslot);
        hslot *= 2;
        hpos = G.pos_of(x, y);
        hcell = (x + 2) + (y + 2) * W2;
        sc[hcell] = I.buf[bit_of(I.par[0], tile)][0][mx + (int64_t)my * nx];
    }
    // ... and of the ring outside or the edge inside: its owner (own: region tile + 1, 0 outside), its place
    int rpos = -1, rx1 = 0, ry1 = 0, own = 0;
    if (tid < nr + ne) {
        int x, y;
        if (tid < nr) {
            outer_cell<1>(tid, w, h, &x, &y);
            rpos = G.pos_of(x, y);
        } else {
            TileRing<TB>::cell(tid - nr, &x, &y, w, h);
            own = 1 + x / TB + y / TB * kx;
            rpos = (x / TB + 2) + (y / TB + 2) * PW;
        }
        rx1 = x + 1;
        ry1 = y + 1;
        if (!own && !regular) {  // a sleeping owner's stored potential
            const int mx = map_index(x0 + x, nx, G.bcx), my = map_index(y0 + y, ny, G.bcy);
            smu[rx1 + ry1 * W1] = TileRing<TB>::stale(mu_store, mx / TB + (my / TB) * ntx, mx, my, nx, ny);
        }
    }
    __syncthreads();
    if (!regular)  // the stored rings of the region's own tiles (read while they sleep)
        for (int j = 0; j < nk; j++) {
            const ResTile& T = tiles[j];
            for (int k = tid; k < TileRing<TB>::size(T.w, T.h); k += nthr) {
                int lx, ly;
                TileRing<TB>::cell(k, &lx, &ly, T.w, T.h);
                smu[(T.x + lx + 1) + (T.y + ly + 1) * W1] = mu_store[(int64_t)T.t * TileRing<TB>::N + k];
            }
        }
    __syncthreads();

    const int grp = tid / NT, gn = nthr / NT;  // NT threads work on a tile at a time
    const int tx = (tid % NT) % TB, ty = (tid % NT) / TB;
    auto strip = [&](const double* s, int stride, int x, int y, double (&out)[R], double (&c)[R]) {
        double L[R + 2], M[R + 2], Rt[R + 2];
#pragma unroll
        for (int r = 0; r < R + 2; r++) {
            const double* q = s + x + (y - 1 + r) * stride;
            L[r] = q[-1];
            M[r] = q[0];
            Rt[r] = q[1];
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            const double s1 = (Rt[r + 1] + L[r + 1]) + (M[r + 2] + M[r]);
            if (NINE) {
                const double s2 = (Rt[r + 2] + L[r + 2]) + (Rt[r] + L[r]);
                out[r] = ((4.0 * s1 + s2) - 20.0 * M[r + 1]) * inv;
            } else {
                out[r] = (s1 - 4.0 * M[r + 1]) * inv;
            }
            c[r] = M[r + 1];
        }
    };
    // mu of tile j but for the region's edge cells (their halo may be on its way)
    auto tile_mu = [&](int j, int* f) {
        const ResTile& T = tiles[j];
        double lc[R], c[R];
        int flag = 0;
        // rows past a partial tile read other window rows, and are not used
        const int yb = T.y + ty * R;
        if (tx < T.w && ty * R < T.h) {
            strip(sc, W2, T.x + tx + 2, yb + 2, lc, c);
#pragma unroll
            for (int r = 0; r < R; r++) {
                const int x = T.x + tx, y = yb + r;
                if (ty * R + r < T.h && x > 0 && x < w - 1 && y > 0 && y < h - 1) {
                    smu[(x + 1) + (y + 1) * W1] = (c[r] * c[r] * c[r] - c[r]) - kappa * lc[r];
                    flag |= fabs(lc[r]) > eps;
                }
            }
        }
        const unsigned long long v = __ballot(flag);
        if (lane == 0 && v) f[j] = 1;
    };

    // frame slots of the thread's cells of the group's first tile (-1: not published)
    int slot0[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        slot0[r] = -1;
        if (grp < nk) {
            const ResTile& T = tiles[grp];
            if (tx < T.w && ty * R + r < T.h) slot0[r] = frame_slot(T.x + tx, T.y + ty * R + r, w, h);
        }
    }

#pragma unroll 1
    for (int s = 0; s < n; s++) {
        const uint32_t seq = X.base + (uint32_t)s;
        const uint64_t* fin = X.frame + (s & 1) * plane;
        uint64_t* fout = X.frame + ((s & 1) ^ 1) * plane;
        int* f = fire[s % 3];
        const int* fp = fire[(s + 2) % 3];
        // 1. mu of the tiles that certainly run
        for (int j = grp; j < nk; j += gn)
            if (regular || (s > 0 && fp[j])) tile_mu(j, f);
        // 2. the frames of the tiles outside that ran, the detector bits around
        if (s > 0) {
            const uint64_t ran = sact[(s & 1) ^ 1];
            if (hpos >= 0 && ((ran >> hpos) & 1ull)) sc[hcell] = wait_double(fin + hslot, seq, X, &gone[s & 1]);
            if (tid >= nthr - 64) {
                const uint64_t exist = __ballot(near >= 0);
                uint64_t m = exist;
                if (!regular) {
                    const int own_tile = G.inside(lane);
                    int b = 0;
                    if (near >= 0)
                        b = own_tile >= 0 ? fp[own_tile]
                                          : wait_flag(X.flag + (int64_t)((s & 1) ^ 1) * I.nt + near, seq, X, &gone[s & 1]);
                    m = G.dilate(__ballot(b), exist);
                }
                if (lane == 0) sact[s & 1] = m;
            }
        }
        if (tid < kResMaxTiles) fire[(s + 1) % 3][tid] = 0;
        lds_barrier();
        // the same in every wave: the next write of this word is past the next step's barriers
        const int quit = gone[s & 1];
        const uint64_t act = sact[s & 1];
        auto runs = [&](int j) { return (act >> tiles[j].pos) & 1ull; };
        // 3. mu of tiles a neighbour woke, of the region's edge, of the ring of running tiles outside
        for (int j = grp; j < nk; j += gn)
            if (!regular && !(s > 0 && fp[j]) && runs(j)) tile_mu(j, f);
        if (rpos >= 0 && ((act >> rpos) & 1ull)) {
            const double* q = sc + (rx1 + 1) + (ry1 + 1) * W2;
            const double s1 = (q[1] + q[-1]) + (q[W2] + q[-W2]);
            double lc;
            if (NINE) {
                const double s2 = (q[W2 + 1] + q[W2 - 1]) + (q[-W2 + 1] + q[-W2 - 1]);
                lc = ((4.0 * s1 + s2) - 20.0 * q[0]) * inv;
            } else {
                lc = (s1 - 4.0 * q[0]) * inv;
            }
            const double cv = q[0];
            smu[rx1 + ry1 * W1] = (cv * cv * cv - cv) - kappa * lc;
            if (own && fabs(lc) > eps) f[own - 1] = 1;
        }
        lds_barrier();
        // 4. c' into the window, the region's frame to the others
        for (int j = grp; j < nk; j += gn) {
            if (!runs(j)) continue;
            const ResTile& T = tiles[j];
            if (tx < T.w && ty * R < T.h) {
                double lm[R], mu[R];
                const int yb = T.y + ty * R, x = T.x + tx;
                strip(smu, W1, x + 1, yb + 1, lm, mu);
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const int y = yb + r;
                    if (ty * R + r < T.h) {
                        double* q = sc + (x + 2) + (y + 2) * W2;
                        const double cv = *q, change = dt * (mob * lm[r] - rg * (cv - cbar)), cn = cv + change;
                        *q = cn;
                        const int slot = j == grp ? slot0[r] : frame_slot(x, y, w, h);
                        if (slot >= 0 && s + 1 < n) put_double(fout + 2 * ((int64_t)rgn * X.slots + slot), cn, seq + 1);
                    }
                }
            }
        }
        if (tid < nk) {
            ResTile& T = tiles[tid];
            const bool ran = runs(tid);
            const int any = !regular && ran ? f[tid] : 0;
            if (!regular && s + 1 < n)
                xput(X.flag + (int64_t)(s & 1) * I.nt + T.t, (uint64_t)(seq + 1) << 32 | (uint32_t)any);
            f[tid] = any;
            if (ran) {
                T.runs++;
                T.last = any;
                if (I.hist_cap > 0) {
                    const int64_t step = I.ctr[0] + s;
                    if (step < I.hist_cap) atomicAdd((int*)&I.hist[2 * step], 1);
                }
            }
        }
        lds_barrier();
        if (quit) break;
    }

    if (gone[0] | gone[1]) {
        if (tid == 0) resident_give_up(X);
        return;
    }
    if (!regular) {
        // rings to store: of tiles that ran but did not fire when they last did
        bool rings = false;
        for (int j = 0; j < nk; j++) rings |= tiles[j].runs > 0 && !tiles[j].last;
        if (tid == 0) sact[0] = resident_all_done(X, rings);
        __syncthreads();
        if (!sact[0]) return;
    }

    // ---- the state the other paths read: the cells into the buffer that was not
    //      current (others may still read this launch's start from that one), the
    //      rings, the per-tile bytes of the last step, the update counts
    for (int j = 0; j < nk; j++) {
        const ResTile& T = tiles[j];
        if (T.runs > 0) {
            gdouble* out = I.buf[T.par ^ 1][0];
            for (int k = tid; k < T.w * T.h; k += nthr) {
                const int x = T.x + k % T.w, y = T.y + k / T.w;
                out[(x0 + x) + (int64_t)(y0 + y) * nx] = sc[(x + 2) + (y + 2) * W2];
            }
            if (!regular && !T.last)
                for (int k = tid; k < TileRing<TB>::size(T.w, T.h); k += nthr) {
                    int lx, ly;
                    TileRing<TB>::cell(k, &lx, &ly, T.w, T.h);
                    mu_store[(int64_t)T.t * TileRing<TB>::N + k] = smu[(T.x + lx + 1) + (T.y + ly + 1) * W1];
                }
        }
        if (tid == 0) {
            I.dF[n & 1][T.t] = (uint8_t)fire[(n + 2) % 3][j];
            I.dP[n & 1][T.t] = (uint8_t)(T.par ^ (T.runs > 0));
            I.druns[T.t] = T.runs;
        }
    }
}

}  // namespace dba
