// k_kh.h - fused DBA step for 2D compressible Euler (Kelvin-Helmholtz):
// MUSCL-Hancock with central gradients, half-step predictor and Rusanov fluxes.
//
// Reference counterpart: getPrimitive_wakeup -> extrap_in_time_wakeup ->
// calc_flux_wakeup -> apply_flux_wakeup -> Wakeup_Next
// (example_Kelvin_Helmholtz/KH_DBA.cu:418-985), conserved variant
// example_Kelvin_Helmholtz/Conserved/KH_DBA.cu:832-955. Same arithmetic
// (getFlux :662-697, extrapolateInSpaceToFace :630-660, applyFluxes :818-841),
// generalised to a gas gamma, a CFL time step and reflective y walls (mirrored
// ghost cells with the normal velocity negated).
//
// The reference reads the primitives, gradients, primes and fluxes that
// sleeping neighbours left behind. Only a tile's edges are ever read that way,
// so each awake tile stores exactly those: primitives on its ring, (primes,
// x-gradients) on its left column, (primes, y-gradients) on its bottom row, the
// x-face flux of its right column and the y-face flux of its top row.
// Everything else is recomputed in LDS from the conserved state of the tile
// and its neighbours (2-cell halo). The stored state is one contiguous record
// per tile (KhEdge), so a tile's edge writes coalesce instead of landing one
// 8-byte value per cache line down its columns.
//
// What bounds it: the VALU instructions it issues (FP64 takes 4.5-5.5 cycles per
// wave instruction here, and a 16 x 16 tile wave issues about 970). So every
// quantity is computed once: one thread per cell holds what its cell gives the
// faces to its right and above in registers, gradients are taken once per cell,
// and divisions by one number share its reciprocal (below). Before that the
// gradients were taken again at every face, each division was a full one and a
// wave issued 2411: 2048^2 with every tile awake 241 -> 187 us per step (the
// 600-step run from the shear layers 69.5 -> 59.6 ms), the reference's 512^2 on
// 8 x 8 tiles 43.0 -> 26.3 us per step. Keeping the next tile's loads in flight
// through the fluxes gave nothing more (187 us), nor did 3 waves per SIMD
// without spills against 4 (2048^2 run 63.4 against 61.7 ms).
#pragma once
#include "common.h"

namespace dba {

// The primitives and the wave speed of a cell with plain divisions, for the
// speeds a CFL run starts from.
struct KhC {
    double g, vol;
};

__device__ __forceinline__ void kh_prims(const KhC& c, double m, double mx, double my, double e, double* r,
                                         double* u, double* v, double* p) {
    const double rho = m / c.vol;
    const double uu = mx / rho / c.vol;
    const double vv = my / rho / c.vol;
    *r = rho;
    *u = uu;
    *v = vv;
    *p = (e / c.vol - 0.5 * rho * (uu * uu + vv * vv)) * (c.g - 1.0);
}

__device__ __forceinline__ double kh_speed(const KhC& c, double r, double u, double v, double p) {
    return sqrt(c.g * p / r) + sqrt(u * u + v * v);
}

// Edge record of a tile, FP64, field-major: ring primitives r, u, v, p (ring
// cell order: bottom row, top row, left column, right column, the columns
// without their corners); left column primes + x-gradients; bottom row primes +
// y-gradients; x-face fluxes (m, u, v, e) of the right column; y-face fluxes of
// the top row.
template <int TB>
struct KhEdge {
    static constexpr int RING = 4 * TB - 4;
    static constexpr int LEFT = 4 * RING;       // [8][TB]: primes, x-gradients by row
    static constexpr int BOTTOM = LEFT + 8 * TB;  // [8][TB]: primes, y-gradients by column
    static constexpr int XF = BOTTOM + 8 * TB;  // [4][TB] by row
    static constexpr int YF = XF + 4 * TB;      // [4][TB] by column
    static constexpr int R = YF + 4 * TB;       // doubles per tile: 40 TB - 16
    // slot of tile-local cell (lx, ly) on the ring, -1 inside
    __device__ __forceinline__ static int ring(int lx, int ly) {
        if (ly == 0) return lx;
        if (ly == TB - 1) return TB + lx;
        if (lx == 0) return 2 * TB + ly - 1;
        if (lx == TB - 1) return 3 * TB - 2 + ly - 1;
        return -1;
    }
    // the cell of ring slot k (the inverse of ring)
    __device__ __forceinline__ static void cell(int k, int* lx, int* ly) {
        if (k < TB) { *lx = k; *ly = 0; }
        else if (k < 2 * TB) { *lx = k - TB; *ly = TB - 1; }
        else if (k < 3 * TB - 2) { *lx = 0; *ly = k - 2 * TB + 1; }
        else { *lx = TB - 1; *ly = k - (3 * TB - 2) + 1; }
    }
};

// ---- Divisions and square roots of the step
//
// The step is bound by the number of VALU instructions it issues, and a
// correctly rounded division (about 12) or square root (about 20) costs most of
// what surrounds it. FAST versions give the same doubles in fewer: the textbook
// sequences (Newton on the hardware reciprocal, the quotient corrected once by
// its exact remainder; Goldschmidt's square root) without the scaling and the
// special cases around them, and with the refined reciprocal shared by every
// division by the same number. Scaling by powers of two changes no rounding while
// nothing under- or overflows, so inside the ranges kh_guard checks the result is
// the correctly rounded one, as without FAST. A tile with any value outside them
// (vacuum, blow-up, NaN) is redone by the FAST = false instance.
template <bool FAST>
__device__ __forceinline__ double kh_rcp(double b) {
    if constexpr (FAST) {
        double y = __builtin_amdgcn_rcp(b);
        y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
        return __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
    } else {
        return 0.0;  // unused
    }
}

// a / b, y = kh_rcp(b)
template <bool FAST>
__device__ __forceinline__ double kh_div(double a, double b, double y) {
    if constexpr (FAST) {
        const double q = a * y;
        return __builtin_fma(__builtin_fma(-b, q, a), y, q);
    } else {
        return a / b;
    }
}

// x >= 0; POS: x is known not to be 0
template <bool FAST, bool POS>
__device__ __forceinline__ double kh_sqrt(double x) {
    if constexpr (FAST) {
        const double y = __builtin_amdgcn_rsq(x);
        double g = x * y, h = y * 0.5;
        const double e = __builtin_fma(-h, g, 0.5);
        h = __builtin_fma(h, e, h);
        g = __builtin_fma(g, e, g);
        g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
        g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
        return POS ? g : (x == 0.0 ? 0.0 : g);
    } else {
        return sqrt(x);
    }
}

// Constants of a step with the reciprocals of what it divides by.
struct KhStep {
    double g, gm1, dt, hdt;    // gamma, gamma - 1, dt, dt / 2
    double dx, vol;            // dy == dx
    double igm1, idx, ivol;    // P2: exact reciprocals of dx and vol; else kh_rcp
    bool sane;                 // every constant within the range the guard assumes
};

// x / d for a constant d of the step. P2: d is a power of two (the spacings and
// the cell area of a power-of-two grid on a unit square), so x * (1/d) rounds the
// same exact real as x / d and gives the same double in every case.
template <bool P2, bool FAST>
__device__ __forceinline__ double kh_cdiv(double x, double d, double y) {
    if constexpr (P2) return x * y;
    else return kh_div<FAST>(x, d, y);
}

// Whether r, p lie in [2^-60, 2^60) and u, v are 0 or in [2^-150, 2^60) in
// magnitude: then no intermediate of the FAST sequences under- or overflows
// anywhere in the step (products of at most four of these, the spacings and dt
// stay within 2^+-1000), except that a face value of r or p may cancel to
// nothing, which the flux checks itself. NaN and infinities fail.
__device__ __forceinline__ bool kh_guard(double r, double u, double v, double p) {
    auto hi = [](double x) { return (unsigned)((unsigned long long)__double_as_longlong(x) >> 32); };
    constexpr unsigned lo60 = (1023u - 60u) << 20, n60 = 120u << 20;
    constexpr unsigned lo150 = (1023u - 150u) << 20, n150 = 210u << 20;
    const bool rp = hi(r) - lo60 < n60 && hi(p) - lo60 < n60;
    const bool uu = (hi(u) & 0x7fffffffu) - lo150 < n150 || u == 0.0;
    const bool vv = (hi(v) & 0x7fffffffu) - lo150 < n150 || v == 0.0;
    return rp && uu && vv;
}

// getPrimitive (example_Kelvin_Helmholtz/KH_DBA.cu:401-405)
template <bool P2, bool FAST>
__device__ __forceinline__ void kh_prim(const KhStep& c, const double (&U)[4], double (&w)[4]) {
    const double r = kh_cdiv<P2, FAST>(U[0], c.vol, c.ivol);
    const double y = kh_rcp<FAST>(r);
    const double u = kh_cdiv<P2, FAST>(kh_div<FAST>(U[1], r, y), c.vol, c.ivol);
    const double v = kh_cdiv<P2, FAST>(kh_div<FAST>(U[2], r, y), c.vol, c.ivol);
    w[0] = r;
    w[1] = u;
    w[2] = v;
    w[3] = (kh_cdiv<P2, FAST>(U[3], c.vol, c.ivol) - 0.5 * r * (u * u + v * v)) * c.gm1;
}

template <bool FAST>
__device__ __forceinline__ double kh_wave_speed(const KhStep& c, const double (&w)[4]) {
    return kh_sqrt<FAST, true>(kh_div<FAST>(c.g * w[3], w[0], kh_rcp<FAST>(w[0]))) +
           kh_sqrt<FAST, false>(w[1] * w[1] + w[2] * w[2]);
}

// getFlux (example_Kelvin_Helmholtz/KH_DBA.cu:662-697) across a face: states
// (rho, velocity across, velocity along, p) of the cell above the face (L) and
// below it (R), in the reference's naming; F = (mass, momentum across, momentum
// along, energy). bad: the FAST sequences do not hold (a density or pressure
// that cancelled to nothing or below).
template <bool FAST>
__device__ __forceinline__ void kh_face(const KhStep& c, const double (&L)[4], const double (&R)[4], double (&F)[4],
                                        bool& bad) {
    const double rL = L[0], uL = L[1], vL = L[2], pL = L[3], rR = R[0], uR = R[1], vR = R[2], pR = R[3];
    if (FAST) {
        constexpr double tiny = 0x1p-200;
        bad |= !(rL > tiny) | !(rR > tiny) | !(pL > tiny) | !(pR > tiny);
    }
    const double eL = kh_div<FAST>(pL, c.gm1, c.igm1) + 0.5 * rL * (uL * uL + vL * vL);
    const double eR = kh_div<FAST>(pR, c.gm1, c.igm1) + 0.5 * rR * (uR * uR + vR * vR);
    const double muL = rL * uL, muR = rR * uR, mvL = rL * vL, mvR = rR * vR;
    const double rho = 0.5 * (rL + rR);
    const double mu = 0.5 * (muL + muR);
    const double mv = 0.5 * (mvL + mvR);
    const double en = 0.5 * (eL + eR);
    const double y = kh_rcp<FAST>(rho);
    const double p = c.gm1 * (en - kh_div<FAST>(0.5 * (mu * mu + mv * mv), rho, y));
    const double cL = kh_sqrt<FAST, true>(kh_div<FAST>(c.g * pL, rL, kh_rcp<FAST>(rL))) + fabs(uL);
    const double cR = kh_sqrt<FAST, true>(kh_div<FAST>(c.g * pR, rR, kh_rcp<FAST>(rR))) + fabs(uR);
    const double hC = (cL >= cR ? cL : cR) * 0.5;
    F[0] = mu - hC * (rL - rR);
    F[1] = (kh_div<FAST>(mu * mu, rho, y) + p) - hC * (muL - muR);
    F[2] = kh_div<FAST>(mu * mv, rho, y) - hC * (mvL - mvR);
    F[3] = kh_div<FAST>((en + p) * mu, rho, y) - hC * (eL - eR);
}

// LDS of a tile: the primitives of the tile and its 2-cell halo; the face values
// to the right of each x face and above each y face. Once the fluxes are in
// registers, the x fluxes take the primitives' space and the y fluxes L's.
template <int TB>
struct KhLds {
    static constexpr int W2 = TB + 4, A2 = W2 * W2, FW = TB + 1, NF = FW * TB;
    double P[4 * A2];
    double L[4 * NF];      // [q][row][face 0..TB]; later the y fluxes [q][face][column]
    double B[4 * NF];      // [q][face][column]
    double E[4 * 2 * TB];  // [q][left column, bottom row]: the outer cells' face values, then the fluxes there
    double red[2][TB * TB / 64], sum[TB * TB / 64 + 1];
    double shift[4][9];
    int vote[TB * TB / 64], bad[TB * TB / 64];
};

// A tile of the list and what its loads need.
struct KhItem {
    CInst* I;
    int t, ti, tj;
    unsigned par, act;  // buffer parity and awake bit of the 3x3 owner tiles, bit d
};

// The halo cells a stencil reads: two cells out on each side, and the corners
// one cell out. Threads H0 .. H0 + 8 TB take the sides, the corners fall to the
// first wave (16 x 16) or to a second round of the only one (8 x 8).
template <int TB>
struct KhHalo {
    static constexpr int NT = TB * TB, NH = 8 * TB + 4, HK = TB == 16 ? 1 : 2;
    // halo cell of this thread's round j, or -1
    __device__ __forceinline__ static int slot(int tid, int j) {
        if (TB == 16) return tid >= 64 && tid < 64 + 8 * TB ? tid - 64 : (tid < 4 ? 8 * TB + tid : -1);
        const int e = tid + j * NT;
        return e < NH ? e : -1;
    }
    // its region coordinates: rows 0, 1, TB + 2, TB + 3, then columns, then corners
    __device__ __forceinline__ static void cell(int e, int& lx, int& ly) {
        if (e < 4 * TB) {
            lx = 2 + e % TB;
            ly = e / TB;
            ly = ly < 2 ? ly : TB + ly;
        } else if (e < 8 * TB) {
            const int k = e - 4 * TB;
            lx = k & 3;
            lx = lx < 2 ? lx : TB + lx;
            ly = 2 + (k >> 2);
        } else {
            lx = (e & 1) ? TB + 2 : 1;
            ly = (e & 2) ? TB + 2 : 1;
        }
    }
};

// The thread's loads of a tile, left in flight: U of its cell and its halo cells
// (U of the owner's current buffer, or the primitives a sleeping owner's ring kept).
template <int TB>
struct KhIn {
    double U[4], h[KhHalo<TB>::HK][4];
};

template <int TB>
__device__ __forceinline__ void kh_load(const KhItem& it, int tid, KhIn<TB>& in) {
    using H = KhHalo<TB>;
    using E = KhEdge<TB>;
    CInst& I = *it.I;
    const int nx = I.nx, ny = I.ny, x0 = it.ti * TB, y0 = it.tj * TB;
    const bool wall = I.bc_y == 2;
    const int pself = (it.par >> 4) & 1;
    const bool plain = it.act == 0x1ffu && (it.par == 0u || it.par == 0x1ffu);  // one buffer, nobody sleeps
    const int64_t base = x0 + (int64_t)y0 * nx;  // uniform; the cell's offset in the tile fits 32 bits
    const unsigned off = (unsigned)(tid % TB + (tid / TB) * nx) * 8u;
#pragma unroll
    for (int q = 0; q < 4; q++) in.U[q] = at_bytes(I.buf[pself][q] + base, off);
#pragma unroll
    for (int j = 0; j < H::HK; j++) {
        const int e = H::slot(tid, j);
        if (e < 0) continue;
        int lx, ly;
        H::cell(e, lx, ly);
        const int mx = map_index(x0 + lx - 2, nx, 0), my = map_index(y0 + ly - 2, ny, wall ? 1 : 0);
        const int64_t gi = mx + (int64_t)my * nx;
        if (plain) {
#pragma unroll
            for (int q = 0; q < 4; q++) in.h[j][q] = I.buf[pself][q][gi];
        } else {
            const int d = nb_dir1<TB, 2>(lx) + 3 * nb_dir1<TB, 2>(ly);
            if ((it.act >> d) & 1u) {
                const bool pp = (it.par >> d) & 1u;
                for (int q = 0; q < 4; q++) in.h[j][q] = (pp ? I.buf[1][q] : I.buf[0][q])[gi];
            } else {
                const int ri = E::ring(mx & (TB - 1), my & (TB - 1));
                const gdouble* er = I.aux[0] + (int64_t)nb_owner2d(I, it.ti, it.tj, d) * E::R + (ri >= 0 ? ri : 0);
                for (int q = 0; q < 4; q++) in.h[j][q] = er[q * E::RING];
            }
        }
    }
}

// Gradients and half-step primes of the cell at k of the LDS primitives: Grad_x /
// Grad_y (example_Kelvin_Helmholtz/KH_DBA.cu:249-275), extrap_in_time (:524-531).
template <int TB, bool P2, bool FAST>
__device__ __forceinline__ void kh_primes(const KhStep& c, const double* sP, int k, double (&pr)[4], double (&gx)[4],
                                          double (&gy)[4]) {
    constexpr int W2 = TB + 4, A2 = W2 * W2;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        gx[q] = kh_cdiv<P2, FAST>((sP[q * A2 + k + 1] - sP[q * A2 + k - 1]) / 2.0, c.dx, c.idx);
        gy[q] = kh_cdiv<P2, FAST>((sP[q * A2 + k + W2] - sP[q * A2 + k - W2]) / 2.0, c.dx, c.idx);
    }
    const double r = sP[k], u = sP[A2 + k], v = sP[2 * A2 + k], p = sP[3 * A2 + k];
    const double ir = kh_div<FAST>(1.0, r, kh_rcp<FAST>(r));
    pr[0] = r - c.hdt * (u * gx[0] + r * gx[1] + v * gy[0] + r * gy[2]);
    pr[1] = u - c.hdt * (u * gx[1] + v * gy[1] + ir * gx[3]);
    pr[2] = v - c.hdt * (u * gx[2] + v * gy[2] + ir * gy[3]);
    pr[3] = p - c.hdt * (c.g * p * (gx[1] + gy[2]) + u * gx[3] + v * gy[3]);
}

// One tile's step: one thread per cell, `in` loaded by kh_load. Each thread keeps
// the values its cell gives the faces on its right and above it in registers and
// puts those for the faces on its left and below it into LDS, so every gradient
// is taken once and a flux needs four LDS reads. The ring cells (the last wave)
// serve the tile's outer faces; what a sleeping neighbour left behind comes from
// its record. The barriers order LDS only, so the tile's stores stay outstanding
// across them.
// FAST: returns false, having stored nothing, when a value leaves the range its
// divisions are exact in.
template <int TB, bool P2, bool FAST>
__device__ __forceinline__ bool kh_tile(const KhItem& it, const KhStep& c, KhLds<TB>& S, KhIn<TB>& in, int tid,
                                        int& any, double& vstale, double& vfresh, double (&part)[4]) {
    using E = KhEdge<TB>;
    using LD = KhLds<TB>;
    using H = KhHalo<TB>;
    constexpr int W2 = LD::W2, A2 = LD::A2, FW = LD::FW, NF = LD::NF, NT = TB * TB, NW = NT / 64, TE = 2 * TB;
    CInst& I = *it.I;
    const int tx = tid % TB, ty = tid / TB, lane = tid & 63, wid = tid >> 6;
    const int t = it.t, nx = I.nx, ny = I.ny;
    const int x0 = it.ti * TB, y0 = it.tj * TB;
    const unsigned par = it.par, act = it.act;
    const bool dba = I.mode != 0, wall = I.bc_y == 2, cfl = I.dt_mode == 1;
    const int ncons = I.ncons;
    const int pself = (par >> 4) & 1;
    const int64_t base = x0 + (int64_t)y0 * nx;
    const unsigned off = (unsigned)(tx + ty * nx) * 8u;
    double* sP = S.P;
    double* sL = S.L;
    double* sB = S.B;
    double* sE = S.E;
    bool bad = FAST && !c.sane;

    // 1. primitives of the cell and of the halo (only ring cells of a sleeping
    //    owner are ever reached)
    vstale = 0.0;
    {
        if (ncons)
            for (int q = 0; q < 4; q++) in.U[q] -= S.shift[q][4];
        double w[4];
        kh_prim<P2, FAST>(c, in.U, w);
        if (FAST) bad |= !kh_guard(w[0], w[1], w[2], w[3]);
        const int k0 = (tx + 2) + (ty + 2) * W2;
#pragma unroll
        for (int q = 0; q < 4; q++) sP[q * A2 + k0] = w[q];
        // the speed at the start of the step; one that is no number does not count
        if (cfl) vstale = fmax(0.0, kh_wave_speed<FAST>(c, w));
    }
#pragma unroll
    for (int j = 0; j < H::HK; j++) {
        const int e = H::slot(tid, j);
        if (e < 0) continue;
        int lx, ly;
        H::cell(e, lx, ly);
        const int gy = y0 + ly - 2;
        double(&h)[4] = in.h[j];
        const int d = nb_dir1<TB, 2>(lx) + 3 * nb_dir1<TB, 2>(ly);
        if ((act >> d) & 1u) {
            if (ncons)
                for (int f = 0; f < 4; f++) h[f] -= S.shift[f][d];
            kh_prim<P2, FAST>(c, h, h);
        } else {
            const int mx = map_index(x0 + lx - 2, nx, 0), my = map_index(gy, ny, wall ? 1 : 0);
            if (E::ring(mx & (TB - 1), my & (TB - 1)) < 0) {
                h[0] = h[3] = 1.0;  // never reached by a stencil
                h[1] = h[2] = 0.0;
            }
        }
        if (FAST) bad |= !kh_guard(h[0], h[1], h[2], h[3]);
        if (wall && (gy < 0 || gy >= ny)) h[2] = -1.0 * h[2];
        const int k = lx + ly * W2;
#pragma unroll
        for (int f = 0; f < 4; f++) sP[f * A2 + k] = h[f];
    }
    lds_barrier();

    // 2. gradients, half-step primes, face values (extrapolateInSpaceToFace,
    //    example_Kelvin_Helmholtz/KH_DBA.cu:630-660: prime -/+ gradient * dx / 2)
    double Rx[4], Ry[4];  // this cell's values at its right and upper face
    int flag = 0;
    {
        double pr[4], gx[4], gy[4];
        kh_primes<TB, P2, FAST>(c, sP, (tx + 2) + (ty + 2) * W2, pr, gx, gy);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const double hx = gx[q] * c.dx / 2.0, hy = gy[q] * c.dx / 2.0;
            sL[q * NF + tx + ty * FW] = pr[q] - hx;
            sB[q * NF + tx + ty * TB] = pr[q] - hy;
            Rx[q] = pr[q] + hx;
            Ry[q] = pr[q] + hy;
        }
        if (dba) {
            const double m = I.metric_kind == 1 ? fabs(gx[0]) + fabs(gy[0])
                                                : fabs(gx[0]) + fabs(gy[0]) + fabs(gx[3]) + fabs(gy[3]) + fabs(gx[1]) +
                                                      fabs(gy[1]) + fabs(gx[2]) + fabs(gy[2]);
            flag = m > I.thresh_a;
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    // the ring: side 0 left, 1 right, 2 below, 3 above
    const int rt = TB == 16 ? tid - (NT - 64) : tid;
    if (rt >= 0 && rt < 4 * TB) {
        const int side = rt / TB, i = rt % TB;
        const int d = side == 0 ? 3 : (side == 1 ? 5 : (side == 2 ? 1 : 7));
        // where this cell's face values go: with the tile's own, or (left, below) on their own
        double* dst = side == 1 ? sL + TB + i * FW : (side == 3 ? sB + i + TB * TB : sE + (side >> 1) * TB + i);
        const int ds = (side & 1) ? NF : TE;
        if ((act >> d) & 1u) {
            const int lx = side == 0 ? 1 : (side == 1 ? TB + 2 : 2 + i), ly = side == 2 ? 1 : (side == 3 ? TB + 2 : 2 + i);
            double pr[4], gx[4], gy[4];
            kh_primes<TB, P2, FAST>(c, sP, lx + ly * W2, pr, gx, gy);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const double h = (side < 2 ? gx[q] : gy[q]) * c.dx / 2.0;
                dst[q * ds] = (side & 1) ? pr[q] - h : pr[q] + h;
            }
        } else {
            const gdouble* e = I.aux[0] + (int64_t)nb_owner2d(I, it.ti, it.tj, d) * E::R;
            if (side & 1) {
                // a sleeping right (upper) neighbour's left column (bottom row): its
                // stored primes and gradients
                e += (side == 1 ? E::LEFT : E::BOTTOM) + i;
                for (int q = 0; q < 4; q++) dst[q * ds] = e[q * TB] - e[(4 + q) * TB] * c.dx / 2.0;
            } else {
                // the fluxes a sleeping left (lower) neighbour kept for its right column (top row)
                e += (side == 0 ? E::XF : E::YF) + i;
                for (int q = 0; q < 4; q++) dst[q * ds] = e[q * TB];
            }
        }
    }
    {
        const unsigned long long vote = __ballot(flag);
        if (lane == 0) S.vote[wid] = vote != 0ull;
    }
    lds_barrier();
    // a tile that did not fire leaves its edge state for its neighbours (one that
    // fired is awake next step, and a record is read only while its owner sleeps)
    any = 0;
#pragma unroll
    for (int w = 0; w < NW; w++) any |= S.vote[w];
    const bool store = dba && !any;

    // 3. fluxes: the right and the upper face of the cell; then the faces of the
    //    left column and the bottom row whose outer cell runs
    double Fx[4], Fy[4];
    {
        double L[4];
#pragma unroll
        for (int q = 0; q < 4; q++) L[q] = sL[q * NF + (tx + 1) + ty * FW];
        kh_face<FAST>(c, L, Rx, Fx, bad);
        __builtin_amdgcn_sched_barrier(0);
        // y faces: the velocity across is v
        const int kb = tx + (ty + 1) * TB;
        const double Lb[4] = {sB[kb], sB[2 * NF + kb], sB[NF + kb], sB[3 * NF + kb]};
        const double Rb[4] = {Ry[0], Ry[2], Ry[1], Ry[3]};
        double F[4];
        kh_face<FAST>(c, Lb, Rb, F, bad);
        Fy[0] = F[0];
        Fy[1] = F[2];
        Fy[2] = F[1];
        Fy[3] = F[3];
    }
    __builtin_amdgcn_sched_barrier(0);
    if (tid < TE) {
        const int y = tid / TB, i = tid % TB;
        if ((act >> (y ? 1 : 3)) & 1u) {
            const double* l = y ? sB + i : sL + i * FW;
            const double* r = sE + tid;
            const int a = 1 + y, b = 2 - y;  // the velocities across and along the face
            const double La[4] = {l[0], l[a * NF], l[b * NF], l[3 * NF]};
            const double Ra[4] = {r[0], r[a * TE], r[b * TE], r[3 * TE]};
            double F[4];
            kh_face<FAST>(c, La, Ra, F, bad);
            sE[tid] = F[0];
            sE[a * TE + tid] = F[1];
            sE[b * TE + tid] = F[2];
            sE[3 * TE + tid] = F[3];
        }
    }
    if (FAST) {
        const unsigned long long vote = __ballot(bad);
        if (lane == 0) S.bad[wid] = vote != 0ull;
    }
    lds_barrier();
    if (FAST) {
        int b = 0;
#pragma unroll
        for (int w = 0; w < NW; w++) b |= S.bad[w];
        if (b) return false;
    }
    if (store) {
        gdouble* e = I.aux[0] + (int64_t)t * E::R;
        for (int k = tid; k < E::RING; k += NT) {
            int lx, ly;
            E::cell(k, &lx, &ly);
            const int q = (lx + 2) + (ly + 2) * W2;
            for (int f = 0; f < 4; f++) e[f * E::RING + k] = sP[f * A2 + q];
        }
        // left column: primes and x gradients; bottom row: primes and y gradients
        if (tid < 2 * TB) {
            const int half = tid / TB, i = tid % TB;
            double pr[4], gx[4], gy[4];
            kh_primes<TB, P2, FAST>(c, sP, (half == 0 ? 2 : 2 + i) + (half == 0 ? 2 + i : 2) * W2, pr, gx, gy);
            gdouble* r = e + (half == 0 ? E::LEFT : E::BOTTOM) + i;
            for (int q = 0; q < 4; q++) {
                r[q * TB] = pr[q];
                r[(4 + q) * TB] = half == 0 ? gx[q] : gy[q];
            }
        }
        if (tx == TB - 1)
            for (int q = 0; q < 4; q++) e[E::XF + q * TB + ty] = Fx[q];
        if (ty == TB - 1)
            for (int q = 0; q < 4; q++) e[E::YF + q * TB + tx] = Fy[q];
        lds_barrier();  // the primitives' last reads
    }
    // the cell's state again (from the caches) rather than held in registers through the fluxes
    double U[4];
#pragma unroll
    for (int q = 0; q < 4; q++) U[q] = at_bytes(I.buf[pself][q] + base, off);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        sP[q * NF + tx + ty * TB] = Fx[q];
        sL[q * NF + tx + ty * TB] = Fy[q];
    }
    lds_barrier();

    // 4. apply the fluxes (applyFluxes, example_Kelvin_Helmholtz/KH_DBA.cu:839-840)
    const double dtdx = c.dt * c.dx;
    if (ncons)
        for (int q = 0; q < 4; q++) U[q] -= S.shift[q][4];
    {
        const double* fx = tx > 0 ? sP + (tx - 1) + ty * TB : sE + ty;
        const double* fy = ty > 0 ? sL + tx + (ty - 1) * TB : sE + TB + tx;
        const int sx = tx > 0 ? NF : TE, sy = ty > 0 ? NF : TE;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            part[q] = dtdx * (-1.0 * Fx[q] + fx[q * sx] - 1.0 * Fy[q] + fy[q * sy]);
            U[q] += part[q];
            at_bytes(I.buf[pself ^ 1][q] + base, off) = U[q];
        }
    }
    vfresh = 0.0;
    if (cfl) {
        double w[4];
        kh_prim<P2, FAST>(c, U, w);
        if (!FAST || kh_guard(w[0], w[1], w[2], w[3])) {
            vfresh = kh_wave_speed<FAST>(c, w);
        } else {
            kh_prim<P2, false>(c, U, w);
            vfresh = fmax(0.0, kh_wave_speed<false>(c, w));
        }
    }
    return true;
}

// The tile redone with the plain divisions: a function of its own, so its
// registers do not count against the kernel's (inlined it cost 8% of the step).
template <int TB, bool P2>
__device__ __noinline__ void kh_tile_plain(KhItem it, KhStep c, KhLds<TB>* S, int tid, int* any, double* vstale,
                                           double* vfresh, double* part) {
    KhIn<TB> in;
    double p[4];
    kh_load<TB>(it, tid, in);
    kh_tile<TB, P2, false>(it, c, *S, in, tid, *any, *vstale, *vfresh, p);
    for (int q = 0; q < 4; q++) part[q] = p[q];
}

template <int TB, bool P2>
__global__ __launch_bounds__(TB* TB) __attribute__((amdgpu_waves_per_eu(4))) void kh_step_kernel(const WorkList wl) {
    __shared__ KhLds<TB> S;
    WorkCursor cur;
    Fold FO;
    work_begin(wl, cur, true);
    constexpr bool FOLD = TB == 8;
    const int total = work_open<FOLD>(wl, FO);
    // opaque to the compiler, so that what follows from the thread index alone is
    // worked out per tile instead of being kept in registers across the tiles
    auto thread = [] {
        int v = threadIdx.x;
        asm volatile("" : "+v"(v));
        return v;
    };
    for (;;) {
        KhItem it;
        uint64_t rec;
        if (!work_next<FOLD>(wl, FO, cur, total, &it.I, &it.t, &rec)) break;
        CInst& I = *it.I;
        const int ntx = I.ntx, lane = threadIdx.x & 63;
        it.tj = it.t / ntx;
        it.ti = it.t - it.tj * ntx;
        if (rec & kRecValid) {
            it.par = (unsigned)(rec & 0x1ffull);
            it.act = (unsigned)((rec >> 9) & 0x1ffull);
        } else {  // one ballot of the bitmap bits per wave
            const int o = lane < 9 ? nb_owner2d(I, it.ti, it.tj, lane) : it.t;
            const int pb = bit_of(I.par[0], o), ab = I.mode == 0 ? 1 : bit_of(I.a_cur[0], o);
            it.par = (unsigned)(__ballot(pb) & 0x1ffull);
            it.act = (unsigned)(__ballot(ab) & 0x1ffull);
        }
        KhIn<TB> in;
        kh_load<TB>(it, thread(), in);
        KhStep c;
        c.g = I.gas_gamma;
        c.gm1 = c.g - 1.0;
        c.dt = I.dt_mode == 1 ? I.scal[1] : I.dt;
        c.hdt = 0.5 * c.dt;
        c.dx = I.dx;
        c.vol = I.vol;
        c.igm1 = kh_rcp<true>(c.gm1);
        c.idx = kh_rcp<true>(c.dx);  // exact for a power of two
        c.ivol = kh_rcp<true>(c.vol);
        c.sane = c.dx > 0x1p-40 && c.dx < 0x1p40 && c.gm1 > 0x1p-20 && c.gm1 < 0x1p20 && c.dt > 0x1p-60 &&
                 c.dt < 0x1p20;
        if (I.ncons > 0) {
            if (threadIdx.x < 9) {
                const int d = threadIdx.x, o = nb_owner2d(I, it.ti, it.tj, d);
                for (int f = 0; f < 4; f++)
                    S.shift[f][d] = I.scal[8 + f] - I.s_tile[((int64_t)f * 2 + ((it.par >> d) & 1u)) * I.nt + o];
            }
            __syncthreads();
        }
        int any = 0;
        double vstale = 0.0, vfresh = 0.0, part[4];
        const bool ok = kh_tile<TB, P2, true>(it, c, S, in, thread(), any, vstale, vfresh, part);
        if (!ok) {
            __syncthreads();
            int a1;
            double s1, f1, p1[4];
            kh_tile_plain<TB, P2>(it, c, &S, threadIdx.x, &a1, &s1, &f1, p1);
            any = a1;
            vstale = s1;
            vfresh = f1;
            for (int q = 0; q < 4; q++) part[q] = p1[q];
        }
        // 5. detector byte, per-tile speeds, conserved bookkeeping
        if (I.mode != 0 && threadIdx.x == 0) I.nflag[0][it.t] = (uint8_t)any;
        if (I.dt_mode == 1) {
            // both maxima (exact in any order) over the workgroup in one exchange
            vstale = wave_max_down(vstale);
            vfresh = wave_max_down(vfresh);
            if (lane == 0) {
                S.red[0][threadIdx.x >> 6] = vfresh;
                S.red[1][threadIdx.x >> 6] = vstale;
            }
            lds_barrier();
            if (threadIdx.x < 2) {
                double m = S.red[threadIdx.x][0];
#pragma unroll
                for (int w = 1; w < TB * TB / 64; w++) m = fmax(m, S.red[threadIdx.x][w]);
                I.tspeed[threadIdx.x * I.nt + it.t] = m;
            }
        }
        for (int q = 0; q < I.ncons; q++) {
            const double tot = block_sum<TB * TB>(part[q], S.sum);
            if (threadIdx.x == 0) {
                I.tpart[(int64_t)q * I.nt + it.t] = tot;
                I.s_tile[((int64_t)q * 2 + (((it.par >> 4) & 1u) ^ 1u)) * I.nt + it.t] = I.scal[8 + q];
            }
        }
        lds_barrier();
    }
}

// Per-tile wave speeds of the current state (all tiles), so the first step of
// a CFL run has its dt; the finalize then keeps them current.
template <int TB>
__global__ void kh_prime_kernel(const Inst* __restrict__ insts, int slot) {
    CInst& I = ((CInst*)insts)[slot];
    KhC c;
    c.g = I.gas_gamma;
    c.vol = I.vol;
    __shared__ double sred[5];
    for (int t = blockIdx.x; t < I.nt; t += gridDim.x) {
        const int x0 = (t % I.ntx) * TB, y0 = (t / I.ntx) * TB;
        const int pp = bit_of(I.par[0], t);
        double vm = 0.0;
        for (int k = threadIdx.x; k < TB * TB; k += blockDim.x) {
            const int64_t gi = (x0 + k % TB) + (int64_t)(y0 + k / TB) * I.nx;
            double sh[4];
            for (int q = 0; q < 4; q++)
                sh[q] = q < I.ncons ? I.scal[8 + q] - I.s_tile[((int64_t)q * 2 + pp) * I.nt + t] : 0.0;
            double r, u, v, p;
            kh_prims(c, I.buf[pp][0][gi] - sh[0], I.buf[pp][1][gi] - sh[1], I.buf[pp][2][gi] - sh[2],
                     I.buf[pp][3][gi] - sh[3], &r, &u, &v, &p);
            vm = fmax(vm, kh_speed(c, r, u, v, p));
        }
        vm = block_max<256>(vm, sred);
        if (threadIdx.x == 0) {
            I.tspeed[t] = vm;
            I.tspeed[I.nt + t] = vm;
        }
        __syncthreads();
    }
}

__global__ void kh_dt_kernel(const Inst* __restrict__ insts, int slot) {
    CInst& I = ((CInst*)insts)[slot];
    __shared__ double sred[5];
    double vm = 0.0;
    for (int t = threadIdx.x; t < I.nt; t += blockDim.x) vm = fmax(vm, I.tspeed[t]);
    vm = block_max<256>(vm, sred);
    if (threadIdx.x == 0 && I.dt_mode == 1) I.scal[1] = I.cfl * (I.dx / vm);
}

}  // namespace dba
