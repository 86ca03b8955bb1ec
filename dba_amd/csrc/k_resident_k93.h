// k_resident_k93.h - many DBA steps of one K93 dendrite in one cooperative launch,
// phi and T in LDS from the first step to the last (k_resident.h: the exchange and
// why it ends).
//
// A 512^2 step took 5.8 us with one launch per step: like a Cahn-Hilliard step it is
// bound by the gap between launches, the tables and the trip through the caches.
// Here a region of tiles stays in LDS and a step waits for one exchange: phi two
// cells deep, T one, both under one slot and in flight together.
#pragma once
#include "common.h"
#include "k_k93.h"
#include "k_resident.h"

namespace dba {

// LDS bytes of a region of w x h cells: phi with a two-cell halo, T with a one-cell
// one, the two flux components on the region and its ring, eps^2 of the edge cells.
constexpr size_t k93_resident_bytes(int w, int h) {
    return sizeof(double) *
           ((size_t)(w + 4) * (h + 4) + 3 * (size_t)(w + 2) * (h + 2) + (size_t)(2 * (w + h)));
}

// One thread per cell, whose terms stay in registers between the phases.
//
// A step: 1. what needs no halo, for the tiles that fired (a fired tile runs): the
// fluxes and Laplacians of the cells inside the region, m; 2. the halo, the outside
// detector bits; 3. the same for tiles only a neighbour woke, fluxes of the cells of
// a sleeping tile that an awake neighbour's differences reach, and, one thread per
// cell, of the region's edge and ring; 4. phi', T', the frame, the detector. Per cell
// the arithmetic and its order are k93_tile's, so results are bit-identical.
template <int TB>
__global__ __launch_bounds__(1024) void k93_resident_kernel(const Inst* __restrict__ insts, Exchange X, int n, int gx,
                                                            int gy) {
    constexpr int NT = TB * TB;  // threads of a tile
    extern __shared__ __align__(16) double lds[];
    __shared__ ResTile tiles[kResMaxTiles];
    __shared__ int runsT[kResMaxTiles];           // steps that ran the T set (tiles[].runs: the phi set)
    __shared__ int fire[2][3][kResMaxTiles];      // detector bits of set and step s in fire[set][s % 3]
    __shared__ int cells[kResMaxTiles];           // field-set updates
    __shared__ int gone[2];                       // a wait of step s ran out: gone[s & 1]
    __shared__ uint64_t sact[2][2];               // [s & 1][set]: awake positions of step s
    CInst& I = ((CInst*)insts)[0];
    const int tid = threadIdx.x, lane = tid & 63, nthr = blockDim.x;
    const Region<TB> G(I, gx, gy);
    const int nx = G.nx, ntx = G.ntx, kx = G.kx, ky = G.ky, nk = G.nk, w = G.w, h = G.h, PW = G.PW;
    const int x0 = G.x0, y0 = G.y0, nt = I.nt;
    const bool regular = I.mode == 0;
    const int W2 = w + 4, W1 = w + 2;
    const int nh = W2 * (h + 4) - w * h, nr = W1 * (h + 2) - w * h, ne = 2 * w + 2 * h - 4;
    double* sp = lds;                          // phi at (x, y): sp[x + 2 + (y + 2) W2]
    double* sT = sp + (size_t)W2 * (h + 4);    // T, Fx, Fy at (x, y): [x + 1 + (y + 1) W1]
    double* sFx = sT + (size_t)W1 * (h + 2);
    double* sFy = sFx + (size_t)W1 * (h + 2);
    double* sE2 = sFy + (size_t)W1 * (h + 2);  // eps^2 of edge cell k (TileRing's order)
    const int64_t plane = (int64_t)gridDim.x * X.slots * 4;
    const int near = G.near(lane);  // the tile at this lane's position
    const int own = G.inside(lane);

    // ---- tables and the state the launch starts from
    if (tid < nk) {
        const int i = tid % kx, j = tid / kx;
        ResTile& T = tiles[tid];
        T.t = (G.ti0 + i) + (G.tj0 + j) * ntx;
        T.x = i * TB;
        T.y = j * TB;
        T.w = min(TB, w - T.x);
        T.h = min(TB, h - T.y);
        T.par = bit_of(I.par[0], T.t) | bit_of(I.par[1], T.t) << 1;
        T.runs = 0;
        T.pos = (i + 2) + (j + 2) * PW;
        runsT[tid] = cells[tid] = 0;
        for (int q = 0; q < 3; q++) fire[0][q][tid] = fire[1][q][tid] = 0;
    }
    if (tid < 64) {
        for (int q = 0; q < 2; q++) {
            const uint64_t m = __ballot(near >= 0 && (regular || bit_of(I.a_cur[q], near)));
            if (lane == 0) {
                sact[0][q] = m;
                sact[1][q] = 0ull;
            }
        }
        if (lane == 0) {
            gone[0] = resident_state(X) == kResGivenUp;
            gone[1] = 0;
        }
    }
    for (int k = tid; k < w * h; k += nthr) {
        const int x = k % w, y = k / w, t = (G.ti0 + x / TB) + (G.tj0 + y / TB) * ntx;
        const int64_t g = (x0 + x) + (int64_t)(y0 + y) * nx;
        sp[(x + 2) + (y + 2) * W2] = I.buf[bit_of(I.par[0], t)][0][g];
        sT[(x + 1) + (y + 1) * W1] = I.buf[bit_of(I.par[1], t)][1][g];
    }
    // this thread's cell of the halo: where it is published, the tile position of its
    // owner, its place in phi and, within the ring, in T
    int hslot = 0, hpos = -1, hphi = 0, hT = -1;
    if (tid < nh) {
        int x, y, mx, my, tile;
        outer_cell<2>(tid, w, h, &x, &y);
        G.source(x, y, X.slots, &mx, &my, &tile, &hslot);
        hslot *= 4;
        hpos = G.pos_of(x, y);
        hphi = (x + 2) + (y + 2) * W2;
        if (x >= -1 && x <= w && y >= -1 && y <= h) hT = (x + 1) + (y + 1) * W1;
        const int64_t g = mx + (int64_t)my * nx;
        sp[hphi] = I.buf[bit_of(I.par[0], tile)][0][g];
        if (hT >= 0) sT[hT] = I.buf[bit_of(I.par[1], tile)][1][g];
    }
    // ... and of the ring outside or the edge inside
    int fx_x = 0, fx_y = 0;
    if (tid < nr) outer_cell<1>(tid, w, h, &fx_x, &fx_y);
    else if (tid < nr + ne) TileRing<TB>::cell(tid - nr, &fx_x, &fx_y, w, h);
    __syncthreads();

    const double inv2dx = I.inv2dx, invdx2 = I.invdx2, alpha_pi = I.alpha_pi, gam = I.gamma;
    const double t_eq = I.t_eq, dt_tau = I.dt_tau, dt = I.dt, lk = I.latent_k;
    const double mp = I.thresh_a, mT = I.thresh_b;

    // the thread's cell: tile, place, frame slot, number on the region's edge (-1: not on it)
    const int j = tid / NT, tx = (tid % NT) % TB, ty = (tid % NT) / TB;
    int x = 0, y = 0, slot = -1, edge = -1, pos = 0;
    bool in = false;
    if (j < nk) {
        const ResTile& T = tiles[j];
        in = tx < T.w && ty < T.h;
        x = T.x + tx;
        y = T.y + ty;
        pos = T.pos;
        if (in) slot = frame_slot(x, y, w, h);
        if (in && (x == 0 || x == w - 1 || y == 0 || y == h - 1)) edge = TileRing<TB>::slot(x, y, w, h);
    }
    double* const qp = sp + (x + 2) + (y + 2) * W2;
    double* const qT = sT + (x + 1) + (y + 1) * W1;
    // eps eps' grad phi of a cell into the flux windows; returns eps^2
    auto flux = [&](int x, int y) {
        const double* q = sp + (x + 2) + (y + 2) * W2;
        const double dx = (q[1] - q[-1]) * inv2dx;
        const double dy = (q[W2] - q[-W2]) * inv2dx;
        double e, a;
        k93_aniso(I, dx, dy, &e, &a);
        const int k = (x + 1) + (y + 1) * W1;
        sFx[k] = a * dx;
        sFy[k] = a * dy;
        return e * e;
    };
    double lap = 0.0, e2 = 0.0, m = 0.0, lapT = 0.0;
    auto laps = [&](bool p, bool T) {
        if (p) lap = ((qp[1] + qp[-1]) + (qp[W2] + qp[-W2]) - 4.0 * qp[0]) * invdx2;
        if (T) lapT = ((qT[1] + qT[-1]) + (qT[W1] + qT[-W1]) - 4.0 * qT[0]) * invdx2;
    };

#pragma unroll 1
    for (int s = 0; s < n; s++) {
        const uint32_t seq = X.base + (uint32_t)s;
        const uint64_t* fin = X.frame + (s & 1) * plane;
        uint64_t* fout = X.frame + ((s & 1) ^ 1) * plane;
        const int cur = s % 3, prev = (s + 2) % 3;
        // 1. what needs no halo, of the tiles that certainly run
        const bool surep = in && (regular || (s > 0 && fire[0][prev][j]));
        const bool sureT = in && (regular || (s > 0 && fire[1][prev][j]));
        if (surep) {
            if (edge < 0) e2 = flux(x, y);
            m = alpha_pi * atan(gam * (t_eq - *qT));
        }
        if (edge < 0) laps(surep, sureT);
        // 2. the cells outside that were advanced, the detector bits around
        if (s > 0) {
            if (hpos >= 0) {
                const uint64_t* q = fin + hslot;
                const bool wp = (sact[(s & 1) ^ 1][0] >> hpos) & 1ull;
                const bool wT = hT >= 0 && ((sact[(s & 1) ^ 1][1] >> hpos) & 1ull);
                if (wp) sp[hphi] = wait_double(q, seq, X, &gone[s & 1]);
                if (wT) sT[hT] = wait_double(q + 2, seq, X, &gone[s & 1]);
            }
            if (tid >= nthr - 64) {
                const uint64_t exist = __ballot(near >= 0);
                uint64_t a = exist, b = exist;
                if (!regular) {
                    int f = 0;
                    if (own >= 0) f = fire[0][prev][own] | fire[1][prev][own] << 1;
                    else if (near >= 0) f = wait_flag(X.flag + (int64_t)((s & 1) ^ 1) * nt + near, seq, X, &gone[s & 1]);
                    a = G.dilate(__ballot(f & 1), exist);
                    b = G.dilate(__ballot(f & 2), exist);
                }
                if (lane == 0) {
                    sact[s & 1][0] = a;
                    sact[s & 1][1] = b;
                }
            }
        }
        if (tid < kResMaxTiles) fire[0][(s + 1) % 3][tid] = fire[1][(s + 1) % 3][tid] = 0;
        lds_barrier();
        const uint64_t actp = sact[s & 1][0], actT = sact[s & 1][1];
        // 3. the rest
        const bool ap = in && ((actp >> pos) & 1ull), aT = in && ((actT >> pos) & 1ull);
        bool reach = ap && !surep;  // the cell's flux is read: by its own tile, or by an awake one beside it
        if (in && !ap) {
            const uint64_t a = actp >> (pos - PW);  // positions from the row below on
            reach = (tx == 0 && ((a >> (PW - 1)) & 1ull)) || (tx == TB - 1 && ((a >> (PW + 1)) & 1ull)) ||
                    (ty == 0 && (a & 1ull)) || (ty == TB - 1 && ((a >> (2 * PW)) & 1ull));
        }
        if (reach && edge < 0) e2 = flux(x, y);
        if (ap && !surep) m = alpha_pi * atan(gam * (t_eq - *qT));
        laps(ap && (edge >= 0 || !surep), aT && (edge >= 0 || !sureT));
        if (tid < nr + ne && actp) {
            const double v = flux(fx_x, fx_y);
            if (tid >= nr) sE2[tid - nr] = v;
        }
        lds_barrier();
        // 4. phi', T', the frame, the detector bits
        int fp = 0, fT = 0;
        if (ap || aT) {
            const double ph = *qp, Tv = *qT;
            double pn = ph;
            uint64_t* q = fout + 4 * ((int64_t)G.rgn * X.slots + slot);
            const bool send = slot >= 0 && s + 1 < n;
            if (ap) {
                const int k = (x + 1) + (y + 1) * W1;
                const double cross = ((sFx[k + W1] - sFx[k - W1]) - (sFy[k + 1] - sFy[k - 1])) * inv2dx;
                const double ee = edge >= 0 ? sE2[edge] : e2;
                const double rhs = (cross + ee * lap) + (ph * (1.0 - ph)) * ((ph - 0.5) + m);
                pn = ph + dt_tau * rhs;
                *qp = pn;
                if (send) put_double(q, pn, seq + 1);
                fp = pn >= mp && pn <= (1.0 - mp);
            }
            if (aT) {
                const double t1 = Tv + dt * lapT;
                const double Tn = ap ? t1 + lk * (pn - ph) : t1;
                *qT = Tn;
                if (send) put_double(q + 2, Tn, seq + 1);
                fT = fabs(Tn - Tv) >= mT;
            }
        }
        if (!regular) {
            const int bits = (__ballot(fp) ? 1 : 0) | (__ballot(fT) ? 2 : 0);
            if (lane == 0 && j < nk) {
                if (bits & 1) fire[0][cur][j] = 1;
                if (bits & 2) fire[1][cur][j] = 1;
            }
        }
        lds_barrier();
        if (tid < nk) {
            ResTile& T = tiles[tid];
            const int rp = (actp >> T.pos) & 1ull, rT = (actT >> T.pos) & 1ull;
            if (!regular && s + 1 < n)
                xput(X.flag + (int64_t)(s & 1) * nt + T.t,
                     (uint64_t)(seq + 1) << 32 | (uint32_t)(fire[0][cur][tid] | fire[1][cur][tid] << 1));
            T.runs += rp;
            runsT[tid] += rT;
            if (rp | rT) cells[tid] += 1 + rp;
            if (I.hist_cap > 0 && (rp | rT)) {
                const int64_t step = I.ctr[0] + s;
                if (step < I.hist_cap) {
                    if (rp) atomicAdd((int*)&I.hist[2 * step], 1);
                    if (rT) atomicAdd((int*)&I.hist[2 * step + 1], 1);
                }
            }
        }
        if (gone[s & 1]) break;  // the same in every wave: the next write of this word is past the next step's barriers
    }
    __syncthreads();
    if (gone[0] | gone[1]) {
        if (tid == 0) resident_give_up(X);
        return;
    }

    // ---- the state the other paths read: per set the cells into the buffer that was
    //      not current (others may still read this launch's start from that one), the
    //      per-tile bytes of the last step, the update counts
    for (int q = 0; q < nk; q++) {
        const ResTile& T = tiles[q];
        const int par = T.par;
        for (int k = tid; k < T.w * T.h; k += nthr) {
            const int lx = T.x + k % T.w, ly = T.y + k / T.w;
            const int64_t g = (x0 + lx) + (int64_t)(y0 + ly) * nx;
            if (T.runs > 0) I.buf[(par & 1) ^ 1][0][g] = sp[(lx + 2) + (ly + 2) * W2];
            if (runsT[q] > 0) I.buf[(par >> 1) ^ 1][1][g] = sT[(lx + 1) + (ly + 1) * W1];
        }
        if (tid == 0) {
            const int last = (n + 2) % 3;
            I.dF[n & 1][T.t] = (uint8_t)fire[0][last][q];
            I.dF[n & 1][nt + T.t] = (uint8_t)fire[1][last][q];
            I.dP[n & 1][T.t] = (uint8_t)((par & 1) ^ (T.runs > 0));
            I.dP[n & 1][nt + T.t] = (uint8_t)((par >> 1) ^ (runsT[q] > 0));
            I.druns[T.t] = cells[q];
        }
    }
}

}  // namespace dba
