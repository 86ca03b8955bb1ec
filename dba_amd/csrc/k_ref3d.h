// k_ref3d.h - fused DBA steps of the reference's own 3D models on 4x4x4
// activation blocks (4x4x1 when nz == 1), periodic.
//
//  * Kobayashi-94 dendrite: Evolve_p(_wakeup) + Evolve_T(_wakeup) + the detector
//    of Wakeup_Next (example_Dendritic_growth/kernel.cu:181-293, 322-574):
//    split p / T sets; regular T = T + dt lapT + p_new - p, DBA T = (T + dt lapT)
//    + (p_new - p) only where p-awake; Pi = 3.14159 (kernel.cu:7).
//  * Ternary Flory-Huggins Model B with reaction: Calc_mu(_wakeup) + detector
//    |lap z| > eps, then Update(_wakeup) + copy-back (example_Reactive_ModelB/
//    kernel.cu:290-763), conserved change capture (example_Reactive_ModelB/
//    Conserved/kernel.cu:630-702). The chemical potentials of sleeping
//    neighbours are the ones they stored when they last ran. Three ways: short lists
//    take two launches with one wave64 per block, longer ones a march up columns of
//    blocks, grids of one plane a kernel of their own.
#pragma once
#include "common.h"
#include "mathf64.h"

namespace dba {

// 27-point isotropic Laplacian (the weights of example_Reactive_ModelB/kernel.cu:
// 333-344) from three planes: with c the centre of a plane, e its four edge
// neighbours and d its four diagonal ones summed,
//     lap = (own(z) + side(z - 1)) + side(z + 1),
//     own = -64/15 c + 7/15 e + d/10,  side = 7/15 c + e/10 + d/30,
// so a march in z reads 8 neighbours per cell and field instead of 26; the block
// kernels evaluate the same expressions.
struct Plane3 {
    double c, own, side;
};

// the sums of one plane around s[0] (row stride RX)
template <int RX>
__device__ __forceinline__ Plane3 plane_sums(const double* s) {
    Plane3 p;
    p.c = s[0];
    const double e = (s[1] + s[-1]) + (s[RX] + s[-RX]);
    const double d = (s[RX + 1] + s[RX - 1]) + (s[-RX + 1] + s[-RX - 1]);
    p.own = __builtin_fma(0.1, d, __builtin_fma(7.0 / 15.0, e, -64.0 / 15.0 * p.c));
    p.side = __builtin_fma(1.0 / 30.0, d, __builtin_fma(0.1, e, 7.0 / 15.0 * p.c));
    return p;
}

// the Laplacian at (x, y, z) of an LDS box with row stride RX and plane stride PZ
template <int RX, int PZ>
__device__ __forceinline__ double lds_lap27(const double* s, int x, int y, int z, double inv_dx2) {
    const double* q = s + x + y * RX + z * PZ;
    const double below = plane_sums<RX>(q - PZ).side, open = plane_sums<RX>(q).own + below;
    return (open + plane_sums<RX>(q + PZ).side) * inv_dx2;
}

template <int TB, int TZ, int H>
__device__ __forceinline__ int nb_dir3(int lx, int ly, int lz) {
    const int a = lx < H ? 0 : (lx < TB + H ? 1 : 2);
    const int b = ly < H ? 0 : (ly < TB + H ? 1 : 2);
    const int c = lz < H ? 0 : (lz < TZ + H ? 1 : 2);
    return a + 3 * b + 9 * c;
}

// ------------------------------------------------------------ Model B (ternary), block kernels
// Two launches per step, like the reference's Calc_mu / Update pair: the first
// computes the chemical potentials of every awake block's own cells into the
// stored-mu arrays (aux 0..2), the second updates x, y, z from the potentials
// of the block and its 1-cell ring. Sleeping neighbours keep the potentials they
// stored when they last ran, so the ring needs no recomputation and each cell's
// logarithms are taken once per step.
//
// One wave per 4x4x4 block, one cell per lane. Both kernels are software
// pipelined over the workgroup's blocks (resolved 64 rounds at a time by
// round_list): while block i computes from LDS, block i+1's box is in flight
// into registers and block i+2's parity words are in flight, so no block waits
// on a dependent chain of loads (worklist -> parities -> box).

// The halo box elements a lane loads (k = lane + 64 i), packed as
// lx | ly << 4 | lz << 8 | neighbour direction << 12 (the same for every block).
template <int TB, int TZ>
struct Box1 {
    static constexpr int WX = TB + 2, WZ = TZ + 2, A = WX * WX * WZ, NH = (A + 63) / 64;
    static constexpr int RX = WX, PZ = WX * WX, AP = A;  // LDS row and plane strides
    int c[NH];
    __device__ __forceinline__ void init(int lane) {
#pragma unroll
        for (int i = 0; i < NH; i++) {
            const int k = lane + i * 64;
            const int lx = k % WX, ly = (k / WX) % WX, lz = k / (WX * WX);
            c[i] = lx | ly << 4 | lz << 8 | nb_dir3<TB, TZ, 1>(lx, ly, lz) << 12;
        }
    }
};

// v in [-1, n] wrapped into [0, n)
__device__ __forceinline__ int wrap1(int v, int n) {
    v = v < 0 ? v + n : v;
    return v >= n ? v - n : v;
}

// Band sweep, for a single instance whose list holds every block (the usual
// case of a fully awake 3D field). Workgroups are dealt to the 8 XCDs
// round-robin by index, so XCD x = b mod 8 owns the band of Cx = ntx*nty/8
// consecutive block columns [x Cx, (x+1) Cx) and sweeps it z-layer by z-layer:
// the band's blocks in (z-block, column) order are dealt round-robin to the
// XCD's S = G/8 workgroups (item i = b/8 + k S). With a grid that is resident
// at once, the XCD's workgroups work on a contiguous run of that order at any
// moment, so a halo plane is still in the XCD's L2 when the blocks on its
// other side need it, and only the two band edges read across XCDs.
// cx = 0 where the grid or the list does not allow it (list order applies).
struct BandSweep {
    int cx, c, per, s, j, base;
};

__device__ __forceinline__ BandSweep band_sweep_setup(const WorkList& w, int total) {
    BandSweep bs{0, 0, 0, 0, 0, 0};
    // one instance (segments are in instance order) whose list is full
    if (w.nseg < 1 || w.segs[w.nseg - 1].inst != 0) return bs;
    const CInst& I = *(const CInst*)w.insts;
    if (total != I.nt) return bs;
    const int G = gridDim.x, C = I.ntx * I.nty;
    if ((G & 7) != 0 || (C & 7) != 0) return bs;
    bs.cx = C >> 3;
    bs.c = C;
    bs.per = I.nt >> 3;
    bs.s = G >> 3;
    bs.j = blockIdx.x >> 3;
    bs.base = (blockIdx.x & 7) * bs.cx;
    return bs;
}

// The sweep's blocks k = round0 .. round0+63 of this workgroup in the RoundList
// form (lane k - round0: item b/8 + k S of its XCD's order).
__device__ __forceinline__ RoundList band_sweep_round(const BandSweep& bs, int round0) {
    const int64_t i = bs.j + (int64_t)(round0 + (int)(threadIdx.x & 63)) * bs.s;
    const bool ok = i < bs.per;
    RoundList L;
    L.inst = 0;
    L.t = ok ? (int)(i / bs.cx) * bs.c + bs.base + (int)(i % bs.cx) : 0;
    L.valid = __ballot(ok);
    return L;
}

// A block of the worklist and what its loads need (all wave-uniform).
struct MbBlock {
    CInst* I;
    int t, x0, y0, z0;
    uint64_t pm;  // parity of the 27 neighbour blocks, bit d = (dx+1) + 3 (dy+1) + 9 (dz+1)
};

template <int TB, int TZ>
__device__ __forceinline__ MbBlock mb_take(const WorkList& w, const RoundList& L, uint64_t& todo) {
    MbBlock b;
    round_take(w, L, todo, &b.I, &b.t);
    CInst& I = *b.I;
    b.x0 = (b.t % I.ntx) * TB;
    b.y0 = ((b.t / I.ntx) % I.nty) * TB;
    b.z0 = (b.t / (I.ntx * I.nty)) * TZ;
    b.pm = 0;
    return b;
}

// Parity of neighbour block `lane` (lanes 0..26): the bitmap word is loaded
// here and the bit taken later (mb_parities_finish), so the load stays in flight.
struct ParityWord {
    uint64_t word;
    int tt;
};

template <int TB, int TZ>
__device__ __forceinline__ ParityWord mb_parities_issue(const MbBlock& b, int lane) {
    CInst& I = *b.I;
    ParityWord p{0ull, 0};
    if (lane < 27) {
        const int dx = lane % 3 - 1, dy = (lane / 3) % 3 - 1, dz = lane / 9 - 1;
        const int mx = wrap1(dx < 0 ? b.x0 - 1 : b.x0 + dx * TB, I.nx);
        const int my = wrap1(dy < 0 ? b.y0 - 1 : b.y0 + dy * TB, I.ny);
        const int mz = wrap1(dz < 0 ? b.z0 - 1 : b.z0 + dz * TZ, I.nz);
        p.tt = mx / TB + (my / TB) * I.ntx + (mz / TZ) * I.ntx * I.nty;
        p.word = I.par[0][p.tt >> 6];
    }
    return p;
}

// One ballot gathers the 27 bits; with conserved DBA lanes 0..26 also store each
// neighbour's pending shift S_f - epoch in sshift (read after a barrier).
__device__ __forceinline__ void mb_parities_finish(MbBlock& b, const ParityWord& p, int lane,
                                                   double (*sshift)[27]) {
    CInst& I = *b.I;
    const int bit = lane < 27 ? (int)((p.word >> (p.tt & 63)) & 1ull) : 0;
    b.pm = __ballot(bit);
    if (lane < 27)
        for (int f = 0; f < I.ncons; f++)
            sshift[f][lane] = I.scal[8 + f] - I.s_tile[((int64_t)f * 2 + bit) * I.nt + p.tt];
}

template <int TB, int TZ>
__device__ __forceinline__ int64_t mb_box_index(const MbBlock& b, int c) {
    CInst& I = *b.I;
    const int lx = c & 15, ly = (c >> 4) & 15, lz = (c >> 8) & 15;
    return wrap1(b.x0 + lx - 1, I.nx) + (int64_t)wrap1(b.y0 + ly - 1, I.ny) * I.nx +
           (int64_t)wrap1(b.z0 + lz - 1, I.nz) * ((int64_t)I.nx * I.ny);
}

// A block whose 1-cell box needs no periodic wrap addresses the box as one
// uniform base plus a per-lane offset (the same for every such block of the
// instance): no wrap selects and no 64-bit index arithmetic per element.
template <int TB, int TZ>
__device__ __forceinline__ bool mb_interior(const MbBlock& b) {
    CInst& I = *b.I;
    return b.x0 > 0 && b.x0 + TB < I.nx && b.y0 > 0 && b.y0 + TB < I.ny && b.z0 > 0 && b.z0 + TZ < I.nz &&
           (int64_t)I.nx * I.ny < (1 << 28);
}

// uniform index of the box corner (x0-1, y0-1, z0-1) of an interior block
__device__ __forceinline__ int64_t mb_box_base(const MbBlock& b) {
    CInst& I = *b.I;
    return (b.x0 - 1) + (int64_t)(b.y0 - 1) * I.nx + (int64_t)(b.z0 - 1) * ((int64_t)I.nx * I.ny);
}

// per-lane offset of packed box element c from the box corner
__device__ __forceinline__ int mb_box_offset(int c, int nx, int nxy) {
    return (c & 15) + ((c >> 4) & 15) * nx + ((c >> 8) & 15) * nxy;
}

template <int TB, int TZ>
__device__ __forceinline__ int64_t mb_own_index(const MbBlock& b, int lane) {
    CInst& I = *b.I;
    const int lx = lane % TB, ly = (lane / TB) % TB, lz = lane / (TB * TB);
    return (b.x0 + lx) + (int64_t)(b.y0 + ly) * I.nx + (int64_t)(b.z0 + lz) * ((int64_t)I.nx * I.ny);
}

// The chemical potentials of a cell (example_Reactive_ModelB/kernel.cu:557-587)
// from x, y, z, phi, the logarithms and the three Laplacians, in parts: what the
// three share (the solvent's terms), then each one's own. The quotients by r_x, r_y and
// r_z are rounded to nearest, from reciprocals the host takes once; the constant of the
// gel term is one quotient on the host, so the term rounds three times, as
// p_gel phi phi / (2 (1 - z_crit)) does. FIN: the logarithms are finite.
template <bool FIN>
__device__ __forceinline__ double mb_over(double a, double b, double y) {
    return FIN ? quotient(a, b, y) : quotient_any(a, b, y);
}

__device__ __forceinline__ double mb_shared(CInst& I, double X, double Y, double Z, double logB) {
    return -(I.chi_xb * X + I.chi_yb * Y + I.chi_zb * Z) - logB;
}

template <bool FIN>
__device__ __forceinline__ double mb_mu_x(CInst& I, double Y, double Z, double B, double com, double logX, double lap) {
    return (I.mb_cx + I.chi_xy * Y + I.chi_xz * Z + I.chi_xb * B + com + mb_over<FIN>(logX, I.r_x, I.mb_irx)) -
           I.epsx_sq * lap;
}

template <bool FIN>
__device__ __forceinline__ double mb_mu_y(CInst& I, double X, double Z, double B, double com, double logY, double lap) {
    return (I.mb_cy + I.chi_xy * X + I.chi_yz * Z + I.chi_yb * B + com + mb_over<FIN>(logY, I.r_y, I.mb_iry)) -
           I.epsy_sq * lap;
}

template <bool FIN>
__device__ __forceinline__ double mb_mu_z(CInst& I, double X, double Y, double B, double com, double logZ, double lap,
                                          double phi) {
    return (I.mb_cz + I.chi_xz * X + I.chi_yz * Y + I.chi_zb * B + com + mb_over<FIN>(logZ, I.r_z, I.mb_irz) -
            I.mb_gel * phi * phi) - I.epsz_sq * lap - I.mb_lk;
}

// The changes of x, y, z of a cell (example_Reactive_ModelB/kernel.cu:419-432):
// dt v_f (mob_f lap mu_f -/+ the reaction)
__device__ __forceinline__ void mb_change(CInst& I, double dfx, double dfy, double dfz, double lx_, double ly_,
                                          double lz_, double (&ch)[3]) {
    const double R = I.k_0 * (exp(I.n_exp * I.v_x * dfx + I.m_exp * I.v_y * dfy) - exp(I.v_z * dfz));
    ch[0] = I.dt * I.v_x * (I.mob_x * lx_ - I.n_exp * R);
    ch[1] = I.dt * I.v_y * (I.mob_y * ly_ - I.m_exp * R);
    ch[2] = I.dt * I.v_z * (I.mob_z * lz_ + R);
}

// ... of the cell at (cx, cy, cz) of an LDS box (field f at sc + f AP); returns
// lap z for the detector. Logarithms first, then one Laplacian at a time: left
// free, the scheduler hoists all 81 LDS reads above the logarithms (250 VGPRs).
template <int RX, int PZ, int AP>
__device__ __forceinline__ double mb_mu_at(CInst& I, const double* sc, int cx, int cy, int cz, double phi,
                                           double (&df)[3]) {
    const int q = cx + cy * RX + cz * PZ;
    const double X = sc[q], Y = sc[AP + q], Z = sc[2 * AP + q];
    const double B = 1.0 - X - Y - Z;
    const double logB = log_f64(B), logX = log_f64(X), logY = log_f64(Y), logZ = log_f64(Z);
    __builtin_amdgcn_sched_barrier(0);
    const double inv_dx2 = I.invdx2;
    const double lx_ = lds_lap27<RX, PZ>(sc, cx, cy, cz, inv_dx2);
    __builtin_amdgcn_sched_barrier(0);
    const double ly_ = lds_lap27<RX, PZ>(sc + AP, cx, cy, cz, inv_dx2);
    __builtin_amdgcn_sched_barrier(0);
    const double lz_ = lds_lap27<RX, PZ>(sc + 2 * AP, cx, cy, cz, inv_dx2);
    __builtin_amdgcn_sched_barrier(0);
    const double com = mb_shared(I, X, Y, Z, logB);
    df[0] = mb_mu_x<false>(I, Y, Z, B, com, logX, lx_);
    df[1] = mb_mu_y<false>(I, X, Z, B, com, logY, ly_);
    df[2] = mb_mu_z<false>(I, X, Y, B, com, logZ, lz_, phi);
    return lz_;
}

template <int RX, int PZ, int AP>
__device__ __forceinline__ void mb_change_at(CInst& I, const double* smu, int cx, int cy, int cz,
                                             double (&ch)[3]) {
    const double inv_dx2 = I.invdx2;
    const int mq = cx + cy * RX + cz * PZ;
    const double dfx = smu[mq], dfy = smu[AP + mq], dfz = smu[2 * AP + mq];
    const double lx_ = lds_lap27<RX, PZ>(smu, cx, cy, cz, inv_dx2);
    __builtin_amdgcn_sched_barrier(0);
    const double ly_ = lds_lap27<RX, PZ>(smu + AP, cx, cy, cz, inv_dx2);
    __builtin_amdgcn_sched_barrier(0);
    const double lz_ = lds_lap27<RX, PZ>(smu + 2 * AP, cx, cy, cz, inv_dx2);
    __builtin_amdgcn_sched_barrier(0);
    mb_change(I, dfx, dfy, dfz, lx_, ly_, lz_, ch);
}

// Calc_mu(_wakeup) + the detector |lap z| > eps (example_Reactive_ModelB/kernel.cu:290-420)
template <int TB, int TZ>
__global__ __launch_bounds__(64) void modelb_mu_kernel(const WorkList wl, int from) {
    using B1 = Box1<TB, TZ>;
    constexpr int A = B1::A, NH = B1::NH, C = TB * TB * TZ, RX = B1::RX, PZ = B1::PZ, AP = B1::AP;
    static_assert(C <= 64, "at most one cell per lane");
    __shared__ double sc[3 * AP];
    __shared__ double sshift[2][kMaxFields][27];

    const int lane = threadIdx.x;
    B1 box;
    box.init(lane);
    double h[NH][3];
    // block q's box (parities known) into h, its own phi into ph
    constexpr uint64_t kAll27 = (1ull << 27) - 1;
    auto load = [&](const MbBlock& q, double& ph) {
        CInst& I = *q.I;
        if (mb_interior<TB, TZ>(q) && (q.pm == 0 || q.pm == kAll27)) {
            // no wrap, and the 27 blocks current in one buffer
            const int p = (int)(q.pm & 1);
            const int64_t base = mb_box_base(q);
            const int nx = I.nx, nxy = I.nx * I.ny;
            const double *b0 = I.buf[p][0] + base, *b1 = I.buf[p][1] + base, *b2 = I.buf[p][2] + base;
#pragma unroll
            for (int i = 0; i < NH; i++) {
                if (lane + i * 64 < A) {
                    const int o = mb_box_offset(box.c[i], nx, nxy);
                    h[i][0] = b0[o];
                    h[i][1] = b1[o];
                    h[i][2] = b2[o];
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < NH; i++) {
                if (lane + i * 64 < A) {
                    const int c = box.c[i];
                    const int64_t gi = mb_box_index<TB, TZ>(q, c);
                    const int pp = (int)(q.pm >> (c >> 12)) & 1;
                    for (int f = 0; f < 3; f++) h[i][f] = I.buf[pp][f][gi];
                }
            }
        }
        if (lane < C) ph = I.buf[(int)(q.pm >> 13) & 1][3][mb_own_index<TB, TZ>(q, lane)];
    };

    __shared__ FoldLds FL;
    Fold FO;
    const int total = work_open(wl, FO, &FL);
    // a list of at least `from` blocks is the march's step
    if (total >= from) return;
    const BandSweep bs = band_sweep_setup(wl, total);
    for (int round0 = 0; (int64_t)round0 * gridDim.x < total; round0 += 64) {
        const RoundList L = bs.cx ? band_sweep_round(bs, round0) : round_list(wl, FO, total, round0);
        uint64_t todo = L.valid;
        if (!todo) continue;
        MbBlock b = mb_take<TB, TZ>(wl, L, todo);
        mb_parities_finish(b, mb_parities_issue<TB, TZ>(b, lane), lane, sshift[0]);
        __syncthreads();
        double phi = 0.0;
        load(b, phi);
        bool has1 = todo != 0;
        MbBlock n1{};
        ParityWord w1{0ull, 0};
        if (has1) {
            n1 = mb_take<TB, TZ>(wl, L, todo);
            w1 = mb_parities_issue<TB, TZ>(n1, lane);
        }
        int slot = 0;
        for (;;) {
            CInst& I = *b.I;
            const int ncons = I.ncons;
            // block b's box into LDS, each value in the current frame
#pragma unroll
            for (int i = 0; i < NH; i++) {
                const int k = lane + i * 64;
                if (k < A) {
                    const int d = box.c[i] >> 12;
                    for (int f = 0; f < 3; f++) {
                        double v = h[i][f];
                        if (f < ncons) v -= sshift[slot][f][d];
                        sc[f * AP + k] = v;
                    }
                }
            }
            __syncthreads();
            double phi_n = 0.0;
            bool has2 = false;
            MbBlock n2{};
            ParityWord w2{0ull, 0};
            if (has1) {
                mb_parities_finish(n1, w1, lane, sshift[slot ^ 1]);
                load(n1, phi_n);
                if (todo) {
                    n2 = mb_take<TB, TZ>(wl, L, todo);
                    w2 = mb_parities_issue<TB, TZ>(n2, lane);
                    has2 = true;
                }
            }

            int flag = 0;
            if (lane < C) {
                const int lx = lane % TB, ly = (lane / TB) % TB, lz = lane / (TB * TB);
                double df[3];
                const double lz_ = mb_mu_at<RX, PZ, AP>(I, sc, lx + 1, ly + 1, lz + 1, phi, df);
                const int64_t gi = mb_own_index<TB, TZ>(b, lane);
                I.aux[0][gi] = df[0];
                I.aux[1][gi] = df[1];
                I.aux[2][gi] = df[2];
                flag = fabs(lz_) > I.thresh_a;
            }
            if (I.mode != 0) {
                const int any = __ballot(flag) != 0ull;
                if (lane == 0) I.nflag[0][b.t] = (uint8_t)any;
            }
            __syncthreads();
            if (!has1) break;
            b = n1;
            phi = phi_n;
            n1 = n2;
            w1 = w2;
            has1 = has2;
            slot ^= 1;
        }
    }
}

// Lane 0 gets the sum over a block's cells (lane x + 4 y + 16 z) in the march's
// order: up in z, then pairs in x, the pairs' pairs, the rows the same way.
__device__ __forceinline__ double mb_block_sum(double v) {
    double s = ((v + __shfl_down(v, 16, 64)) + __shfl_down(v, 32, 64)) + __shfl_down(v, 48, 64);
    s += __shfl_xor(s, 1, 64);
    s += __shfl_xor(s, 2, 64);
    s += __shfl_xor(s, 4, 64);
    s += __shfl_xor(s, 8, 64);
    return s;
}

// Update(_wakeup) + copy-back + conserved change capture
// (example_Reactive_ModelB/kernel.cu:430-560, Conserved/kernel.cu:630-702)
template <int TB, int TZ>
__global__ __launch_bounds__(64) void modelb_update_kernel(const WorkList wl, int from) {
    using B1 = Box1<TB, TZ>;
    constexpr int A = B1::A, NH = B1::NH, C = TB * TB * TZ, RX = B1::RX, PZ = B1::PZ, AP = B1::AP;
    static_assert(C <= 64, "at most one cell per lane");
    __shared__ double smu[3 * AP];

    const int lane = threadIdx.x;
    B1 box;
    box.init(lane);
    double h[NH][3];
    // block q's potentials box into h, its own x, y, z (buffer pq) into vq and
    // their shift epochs into eq (conserved)
    auto load = [&](const MbBlock& q, int pq, double (&vq)[3], double (&eq)[3]) {
        CInst& I = *q.I;
        if (mb_interior<TB, TZ>(q)) {
            const int64_t base = mb_box_base(q);
            const int nx = I.nx, nxy = I.nx * I.ny;
            const double *a0 = I.aux[0] + base, *a1 = I.aux[1] + base, *a2 = I.aux[2] + base;
#pragma unroll
            for (int i = 0; i < NH; i++) {
                if (lane + i * 64 < A) {
                    const int o = mb_box_offset(box.c[i], nx, nxy);
                    h[i][0] = a0[o];
                    h[i][1] = a1[o];
                    h[i][2] = a2[o];
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < NH; i++) {
                if (lane + i * 64 < A) {
                    const int64_t gi = mb_box_index<TB, TZ>(q, box.c[i]);
                    for (int f = 0; f < 3; f++) h[i][f] = I.aux[f][gi];
                }
            }
        }
        if (lane < C) {
            const int64_t gi = mb_own_index<TB, TZ>(q, lane);
            for (int f = 0; f < 3; f++) vq[f] = I.buf[pq][f][gi];
        }
        for (int f = 0; f < I.ncons; f++) eq[f] = I.s_tile[((int64_t)f * 2 + pq) * I.nt + q.t];
    };

    __shared__ FoldLds FL;
    Fold FO;
    const int total = work_open(wl, FO, &FL);
    // a list of at least `from` blocks is the march's step
    if (total >= from) return;
    const BandSweep bs = band_sweep_setup(wl, total);
    for (int round0 = 0; (int64_t)round0 * gridDim.x < total; round0 += 64) {
        const RoundList L = bs.cx ? band_sweep_round(bs, round0) : round_list(wl, FO, total, round0);
        uint64_t todo = L.valid;
        if (!todo) continue;
        MbBlock b = mb_take<TB, TZ>(wl, L, todo);
        int pself = bit_of(b.I->par[0], b.t);
        double v[3] = {0.0, 0.0, 0.0}, e[3] = {0.0, 0.0, 0.0};
        load(b, pself, v, e);
        bool has1 = todo != 0;
        MbBlock n1{};
        uint64_t w1 = 0;
        if (has1) {
            n1 = mb_take<TB, TZ>(wl, L, todo);
            w1 = n1.I->par[0][n1.t >> 6];
        }
        for (;;) {
#pragma unroll
            for (int i = 0; i < NH; i++) {
                const int k = lane + i * 64;
                if (k < A)
                    for (int f = 0; f < 3; f++) smu[f * AP + k] = h[i][f];
            }
            __syncthreads();
            double vn[3] = {0.0, 0.0, 0.0}, en[3] = {0.0, 0.0, 0.0};
            int pn = 0;
            bool has2 = false;
            MbBlock n2{};
            uint64_t w2 = 0;
            if (has1) {
                pn = (int)((w1 >> (n1.t & 63)) & 1ull);
                load(n1, pn, vn, en);
                if (todo) {
                    n2 = mb_take<TB, TZ>(wl, L, todo);
                    w2 = n2.I->par[0][n2.t >> 6];
                    has2 = true;
                }
            }

            CInst& I = *b.I;
            const int ncons = I.ncons;
            double part[3] = {0.0, 0.0, 0.0};
            if (lane < C) {
                const int lx = lane % TB, ly = (lane / TB) % TB, lz = lane / (TB * TB);
                double x[3] = {v[0], v[1], v[2]};
                for (int f = 0; f < ncons; f++) x[f] -= I.scal[8 + f] - e[f];
                double ch[3];
                mb_change_at<RX, PZ, AP>(I, smu, lx + 1, ly + 1, lz + 1, ch);
                const int64_t gi = mb_own_index<TB, TZ>(b, lane);
                I.buf[pself ^ 1][0][gi] = x[0] + ch[0];
                I.buf[pself ^ 1][1][gi] = x[1] + ch[1];
                I.buf[pself ^ 1][2][gi] = x[2] + ch[2];
                part[0] = ch[0];
                part[1] = ch[1];
                part[2] = ch[2];
            }
            for (int f = 0; f < ncons; f++) {
                const double tot = mb_block_sum(part[f]);
                if (lane == 0) {
                    I.tpart[(int64_t)f * I.nt + b.t] = tot;
                    I.s_tile[((int64_t)f * 2 + (pself ^ 1)) * I.nt + b.t] = I.scal[8 + f];
                }
            }
            __syncthreads();
            if (!has1) break;
            b = n1;
            pself = pn;
            for (int f = 0; f < 3; f++) {
                v[f] = vn[f];
                e[f] = en[f];
            }
            n1 = n2;
            w1 = w2;
            has1 = has2;
        }
    }
}

// ------------------------------------------------------------ Model B, column march
// Steps of one 3D Model B instance in which at least `from` blocks are awake (where
// the line lies, and why, stands where the group is built) take
// one launch: a workgroup walks a column of 32 x 12 cells up `nl` layers of
// blocks, plane by plane. Plane p of x, y, z (with a 2-cell halo) goes through
// LDS once; every thread keeps the plane sums of its cell, so plane p completes
// the Laplacians of plane p - 1 and with them its potentials (six waves the
// cells, the other two the ring around them, whose potentials their neighbours
// compute as well); the potentials pass through LDS the same way and complete
// plane p - 2, which is written back. Against the two launches over 8 x 8 x 4
// boxes this replaces, the potentials never go to memory (56 bytes per cell
// instead of the 148 measured), a Laplacian adds 8 neighbours per plane instead
// of 26, and no halo plane is staged twice. What bounds it: FP64 issue (four
// logarithms, two exponentials and six Laplacians per cell, 1.33 x the
// potentials for the ring and (4 nl + 2) / 4 nl for the ends of the strip).
//
// Sleeping blocks: a cell of one presents the potentials it stored when it last
// ran (aux 0..2) and is not written. A block stores its potentials as long as it
// has not fired: plane by plane until the vote of its four waves' cells says so,
// so a block that fires in its first plane stores that plane at most, and one
// that does not fire stores all four, which is all that a later step reads.
// Conserved DBA (CONS): values less the pending shift of their block, and each
// block's change sums (mb_block_sum's order: the block kernels give the same doubles).
struct MbMarch {
    static constexpr int TX = 32, TY = 12, NT = 512;
    static constexpr int CW = TX + 4, CH = TY + 4, CA = CW * CH;  // x, y, z with a 2-cell halo
    static constexpr int MW = TX + 2, MH = TY + 2, MA = MW * MH;  // potentials with their ring
    static constexpr int NI = TX * TY;                            // threads with a cell (six waves)
    static constexpr int NR = MA - NI;                            // threads with a ring cell (of the last two)
    static constexpr int BW = TX / 4 + 2, BH = TY / 4 + 2, NB = BW * BH;  // blocks around a column's layer
    static constexpr int ML = 16, MLC = 8;                        // layers per strip, at most (conserved)
    static_assert(NB <= 64 && NR <= NT - NI && CA <= NT + 64, "one ballot, two ring waves, two loads per thread");
};

// v modulo n for small overshoot of any small n
__device__ __forceinline__ int wrap_any(int v, int n) {
    v %= n;
    return v < 0 ? v + n : v;
}

template <bool CONS>
struct MbMarchLds {
    using M = MbMarch;
    static constexpr int NL = (CONS ? M::MLC : M::ML) + 2;
    double c[3 * M::CA], mu[3 * M::MA];
    uint64_t vote[M::NI / 64];
    uint64_t par[NL], act[NL];                      // parity and awake bits of the blocks of each layer
    double shift[CONS ? NL * M::NB * 3 : 1];        // pending shift of each block
    double part[CONS ? 3 * (M::NI / 64) * 8 : 1];   // change sums of half blocks
};

template <bool CONS>
__global__ __launch_bounds__(MbMarch::NT) __attribute__((amdgpu_waves_per_eu(CONS ? 2 : 4))) void modelb_march_kernel(
    const WorkList wl, int from, int nl, int ncx, int ncy) {
    using M = MbMarch;
    __shared__ MbMarchLds<CONS> S;
    __shared__ FoldLds FL;
    Fold FO;
    const int total = work_open(wl, FO, &FL);
    if (total < from) return;
    CInst& I = *(CInst*)wl.insts;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int nx = I.nx, ny = I.ny, nz = I.nz, ntx = I.ntx, nty = I.nty, ntz = I.ntz;
    const int64_t nxy = (int64_t)nx * ny;
    const bool regular = I.mode == 0;
    const int item = xcd_deal(blockIdx.x, gridDim.x, 0, gridDim.x);
    const int ncol = ncx * ncy, col = item % ncol;
    const int l0 = (item / ncol) * nl, nlay = min(nl, ntz - l0);
    const int x0 = (col % ncx) * M::TX, y0 = (col / ncx) * M::TY;
    const double inv_dx2 = I.invdx2;

    // parity and awake bits of the blocks around each layer l0 - 1 .. l0 + nlay
    for (int k = wid; k < nlay + 2; k += M::NT / 64) {
        const int l = lane < M::NB ? lane : 0;
        const int tt = wrap_any(x0 / 4 + l % M::BW - 1, ntx) + wrap_any(y0 / 4 + l / M::BW - 1, nty) * ntx +
                       wrap_any(l0 + k - 1, ntz) * ntx * nty;
        const gu64 *par0 = I.par[0], *cur0 = I.a_cur[0];
        asm volatile("" : "+s"(par0), "+s"(cur0));
        const uint64_t wp = par0[tt >> 6], wa = cur0[tt >> 6];
        const int pb = (int)((wp >> (tt & 63)) & 1ull);
        const uint64_t pm = __ballot(pb);
        const uint64_t am = regular ? ~0ull : __ballot((int)((wa >> (tt & 63)) & 1ull));
        if (lane == 0) {
            S.par[k] = pm;
            S.act[k] = am;
        }
        if (CONS && lane < M::NB)
#pragma unroll
            for (int f = 0; f < 3; f++)
                S.shift[(k * M::NB + lane) * 3 + f] =
                    I.scal[8 + f] - I.s_tile[((int64_t)f * 2 + pb) * I.nt + tt];
    }
    __syncthreads();
    // the blocks a column owns in a layer, and whether the strip has any to run
    const int bw = min(M::TX, nx - x0) / 4, bh = min(M::TY, ny - y0) / 4;
    uint64_t own = 0ull;
    for (int j = 0; j < bh; j++) own |= ((1ull << bw) - 1ull) << (M::BW * (j + 1) + 1);
    uint64_t run = 0ull;
    for (int k = 1; k <= nlay; k++) run |= S.act[k] & own;
    run = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(run >> 32)) << 32) |
          (uint32_t)__builtin_amdgcn_readfirstlane((int)run);
    if (run == 0ull) return;
    // this thread's loads: region positions tid and, for the last wave, 512 + lane
    const bool two = tid >= M::NT - 64;
    int lbit[2];
    unsigned loff[2];
#pragma unroll
    for (int s = 0; s < 2; s++) {
        const int k = s == 0 ? tid : M::NT + lane, lx = k % M::CW, ly = k / M::CW;
        lbit[s] = ((lx + 2) >> 2) + M::BW * ((ly + 2) >> 2);
        loff[s] = (unsigned)(wrap_any(x0 + lx - 2, nx) + wrap_any(y0 + ly - 2, ny) * nx) * 8u;
    }
    // this thread's cell in the region of the potentials: a cell of the column, or of its ring
    int mx, my;
    if (tid < M::NI) {
        mx = 1 + (tid & 31);
        my = 1 + (tid >> 5);
    } else {
        const int r = min(tid - M::NI, M::NR - 1);
        if (r < 2 * M::MW) {
            mx = r < M::MW ? r : r - M::MW;
            my = r < M::MW ? 0 : M::MH - 1;
        } else {
            const int k = r - 2 * M::MW;
            mx = k < M::TY ? 0 : M::MW - 1;
            my = 1 + (k < M::TY ? k : k - M::TY);
        }
    }
    const bool cell = tid < M::NI;
    const bool mine = cell && mx - 1 < nx - x0 && my - 1 < ny - y0;  // a cell of the grid this column owns
    const int mbit = ((mx + 3) >> 2) + M::BW * ((my + 3) >> 2);
    const unsigned moff = (unsigned)(wrap_any(x0 + mx - 1, nx) + wrap_any(y0 + my - 1, ny) * nx) * 8u;
    const double* sc = S.c + (mx + 1) + (my + 1) * M::CW;
    double* sm = S.mu + mx + my * M::MW;

    double v[2][3];
    auto zof = [&](int p) {  // plane p of the strip (p from -2 to 4 nlay + 1), wrapped
        int z = 4 * l0 + p;
        z = z < 0 ? z + nz : z;
        return z >= nz ? z - nz : z;
    };
    auto bits = [&](const uint64_t* m, int p) {
        const uint64_t w = m[(p + 4) >> 2];
        return ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(w >> 32)) << 32) |
               (uint32_t)__builtin_amdgcn_readfirstlane((int)w);
    };
    // both buffers' plane of field f, and the one lane data picks: pointers held in
    // registers, or the compiler makes a load of the pointer out of the choice
    auto planes = [&](int f, int64_t zo, gdouble*& b0, gdouble*& b1) {
        b0 = I.buf[0][f] + zo;
        b1 = I.buf[1][f] + zo;
        asm volatile("" : "+s"(b0), "+s"(b1));
    };
    auto load = [&](int p) {
        const int64_t zo = (int64_t)zof(p) * nxy;
        const uint64_t pm = bits(S.par, p);
        const bool q0 = (pm >> lbit[0]) & 1ull, q1 = (pm >> lbit[1]) & 1ull;
#pragma unroll
        for (int f = 0; f < 3; f++) {
            gdouble *b0, *b1;
            planes(f, zo, b0, b1);
            v[0][f] = at_bytes(q0 ? b1 : b0, loff[0]);
            if (two) v[1][f] = at_bytes(q1 ? b1 : b0, loff[1]);
        }
    };
    auto deposit = [&](int p) {
        if (CONS) {
            const double* sh = S.shift + ((p + 4) >> 2) * M::NB * 3;
#pragma unroll
            for (int f = 0; f < 3; f++) {
                v[0][f] -= sh[lbit[0] * 3 + f];
                if (two) v[1][f] -= sh[lbit[1] * 3 + f];
            }
        }
#pragma unroll
        for (int f = 0; f < 3; f++) {
            S.c[f * M::CA + tid] = v[0][f];
            if (two) S.c[f * M::CA + M::NT + lane] = v[1][f];
        }
    };

    // of the last plane of x, y, z (c) and of the potentials (m): the value, what it
    // adds to its neighbour planes, its Laplacian without the plane above; and
    // x, y, z of the plane before
    double cv[3], cs[3], co[3], mv[3], ms[3], mo[3], c2[3];
    double part[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int f = 0; f < 3; f++) cv[f] = cs[f] = co[f] = mv[f] = ms[f] = mo[f] = c2[f] = 0.0;
    int fired = 0;
    const int last = 4 * nlay + 1;
    load(-2);
    deposit(-2);
#pragma unroll 1
    for (int p = -2; p <= last; p++) {
        lds_barrier();
        double phi = 0.0;
        if (p >= 0) {
            const int64_t zo = (int64_t)zof(p - 1) * nxy;
            gdouble *b0, *b1;
            planes(3, zo, b0, b1);
            phi = at_bytes((bits(S.par, p - 1) >> mbit) & 1ull ? b1 : b0, moff);
        }
        // on its way until the end of the iteration (after phi: loads return in order)
        if (p < last) load(p + 1);
        // the Laplacians of plane p - 1 and its potentials
        double lap[3], df[3];
        const bool up = p >= 0;
        const bool wakes = (bits(S.act, p - 1 < -2 ? -2 : p - 1) >> mbit) & 1ull;  // this cell's block runs
#pragma unroll
        for (int f = 0; f < 3; f++) {
            const Plane3 n = plane_sums<M::CW>(sc + f * M::CA);
            lap[f] = (co[f] + n.side) * inv_dx2;
            co[f] = n.own + cs[f];
            cs[f] = n.side;
            df[f] = cv[f];
            cv[f] = n.c;
        }
        const double X = df[0], Y = df[1], Z = df[2];
        if (up) {
            if (wakes) {
                const double B = 1.0 - X - Y - Z;
                if (X > 0.0 && Y > 0.0 && Z > 0.0 && B > 0.0) {  // (so all of them are below 1)
                    // one logarithm at a time: together they spill
                    const double com = mb_shared(I, X, Y, Z, log_positive(B));
                    __builtin_amdgcn_sched_barrier(0);
                    df[0] = mb_mu_x<true>(I, Y, Z, B, com, log_positive(X), lap[0]);
                    __builtin_amdgcn_sched_barrier(0);
                    df[1] = mb_mu_y<true>(I, X, Z, B, com, log_positive(Y), lap[1]);
                    __builtin_amdgcn_sched_barrier(0);
                    df[2] = mb_mu_z<true>(I, X, Y, B, com, log_positive(Z), lap[2], phi);
                    __builtin_amdgcn_sched_barrier(0);
                } else {
                    const double com = mb_shared(I, X, Y, Z, log_f64(B));
                    df[0] = mb_mu_x<false>(I, Y, Z, B, com, log_f64(X), lap[0]);
                    df[1] = mb_mu_y<false>(I, X, Z, B, com, log_f64(Y), lap[1]);
                    df[2] = mb_mu_z<false>(I, X, Y, B, com, log_f64(Z), lap[2], phi);
                }
            } else {
                const int64_t zo = (int64_t)zof(p - 1) * nxy;
#pragma unroll
                for (int f = 0; f < 3; f++) df[f] = at_bytes(I.aux[f] + zo, moff);
            }
            if (tid < M::NI + M::NR)
#pragma unroll
                for (int f = 0; f < 3; f++) sm[f * M::MA] = df[f];
            if (cell && !regular) {
                const uint64_t w = __ballot(mine && wakes && fabs(lap[2]) > I.thresh_a);
                if (lane == 0) S.vote[wid] = w;
            }
        }
        lds_barrier();
        if (cell && up) {
            // plane p - 1 of the potentials: stored until the block is known to have fired
            const int q = p - 1;
            if (!regular && mine && q >= 0 && q < 4 * nlay) {
                // the block's cells in this plane: four lanes in two rows, of this wave and its partner
                const uint64_t w = S.vote[wid & ~1] | S.vote[wid | 1];
                const uint64_t m = (0xFull | 0xFull << 32) << (tid & 28);
                fired |= (w & m) != 0ull;
                if (wakes && !fired) {
                    const int64_t zo = (int64_t)zof(q) * nxy;
#pragma unroll
                    for (int f = 0; f < 3; f++) at_bytes(I.aux[f] + zo, moff) = df[f];
                }
                if ((q & 3) == 3) {
                    if (wakes && (tid & 3) == 0 && ((tid >> 5) & 3) == 0)
                        I.nflag[0][(x0 + mx - 1) / 4 + ((y0 + my - 1) / 4) * ntx + (l0 + q / 4) * ntx * nty] =
                            (uint8_t)fired;
                    fired = 0;
                }
            }
            // the changes of plane p - 2
#pragma unroll
            for (int f = 0; f < 3; f++) {
                const Plane3 n = plane_sums<M::MW>(sm + f * M::MA);
                lap[f] = (mo[f] + n.side) * inv_dx2;
                mo[f] = n.own + ms[f];
                ms[f] = n.side;
                df[f] = mv[f];
                mv[f] = n.c;
            }
            if (p >= 2) {
                const int zr = p - 2;
                const bool ran = mine && ((bits(S.act, zr) >> mbit) & 1ull);
                double ch[3];
                mb_change(I, df[0], df[1], df[2], lap[0], lap[1], lap[2], ch);
                if (ran) {
                    const int64_t zo = (int64_t)zof(zr) * nxy;
                    const bool q = (bits(S.par, zr) >> mbit) & 1ull;
#pragma unroll
                    for (int f = 0; f < 3; f++) {
                        gdouble *b0, *b1;
                        planes(f, zo, b0, b1);
                        at_bytes(q ? b0 : b1, moff) = c2[f] + ch[f];
                    }
                }
                if (CONS) {
#pragma unroll
                    for (int f = 0; f < 3; f++) part[f] += ran ? ch[f] : 0.0;
                    if ((zr & 3) == 3) {
#pragma unroll
                        for (int f = 0; f < 3; f++) {
                            double s = part[f];
                            s += __shfl_xor(s, 1, 64);
                            s += __shfl_xor(s, 2, 64);
                            s += __shfl_xor(s, 32, 64);
                            if ((lane & 35) == 0) S.part[(f * (M::NI / 64) + wid) * 8 + (lane >> 2)] = s;
                            part[f] = 0.0;
                        }
                    }
                }
            }
        }
        if (CONS && p >= 2 && ((p - 2) & 3) == 3) {
            lds_barrier();
            // a block's change sums: its two waves' halves
            if (tid < 3 * (M::TY / 4) * 8) {
                const int f = tid / (8 * (M::TY / 4)), r = tid % (8 * (M::TY / 4)), j = r / 8, i = r % 8;
                const int bit = (i + 1) + M::BW * (j + 1), lay = (p - 2) / 4 + 1;
                if (i < bw && j < bh && ((S.act[lay] >> bit) & 1ull)) {
                    const int t = x0 / 4 + i + (y0 / 4 + j) * ntx + (l0 + lay - 1) * ntx * nty;
                    const int b = (int)((S.par[lay] >> bit) & 1ull);
                    const double* h = S.part + (f * (M::NI / 64) + 2 * j) * 8 + i;
                    I.tpart[(int64_t)f * I.nt + t] = h[0] + h[8];
                    I.s_tile[((int64_t)f * 2 + (b ^ 1)) * I.nt + t] = I.scal[8 + f];
                }
            }
        }
        c2[0] = X;
        c2[1] = Y;
        c2[2] = Z;
        // every read of plane p's sums was before the second barrier
        if (p < last) deposit(p + 1);
    }
}

// ------------------------------------------------------------ Model B, one plane
// The march's step of a grid of one plane (nz == 1, blocks of 4 x 4 x 1): a workgroup
// takes 32 x 12 cells, the plane above and the one below are the plane itself, and
// there is nothing to walk. Against the two block kernels, whose waves have a cell
// on 16 of their 64 lanes: bound by the chain of loads and two barriers of a
// workgroup on small grids, by FP64 issue on large ones. Same doubles, same stored
// potentials and detector bytes. us per step, two block kernels -> this: 300^2
// 36 -> 13, conserved 700^2 153 -> 35, 4096^2 2560 -> 514.
template <bool CONS>
struct MbPlaneLds {
    using M = MbMarch;
    double c[3 * M::CA], mu[3 * M::MA];
    uint64_t vote[M::NI / 64];
    uint64_t par, act;                             // parity and awake bits of the blocks around
    double shift[CONS ? M::NB * 3 : 1];            // pending shift of each block
    double part[CONS ? 3 * (M::NI / 64) * 8 : 1];  // change sums of half blocks
};

template <bool CONS>
__global__ __launch_bounds__(MbMarch::NT) __attribute__((amdgpu_waves_per_eu(4))) void modelb_plane_kernel(
    const WorkList wl, int from, int ncx) {
    using M = MbMarch;
    __shared__ MbPlaneLds<CONS> S;
    __shared__ FoldLds FL;
    Fold FO;
    const int total = work_open(wl, FO, &FL);
    if (total < from) return;
    CInst& I = *(CInst*)wl.insts;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int nx = I.nx, ny = I.ny, ntx = I.ntx, nty = I.nty;
    const bool regular = I.mode == 0;
    const int col = xcd_deal(blockIdx.x, gridDim.x, 0, gridDim.x);
    const int x0 = (col % ncx) * M::TX, y0 = (col / ncx) * M::TY;
    const double inv_dx2 = I.invdx2;
    auto block_at = [&](int bit) {  // the block at a bit of the masks
        return wrap_any(x0 / 4 + bit % M::BW - 1, ntx) + wrap_any(y0 / 4 + bit / M::BW - 1, nty) * ntx;
    };

    if (wid == 0) {
        const int tt = block_at(lane < M::NB ? lane : 0);
        const gu64 *par0 = I.par[0], *cur0 = I.a_cur[0];
        asm volatile("" : "+s"(par0), "+s"(cur0));
        const uint64_t wp = par0[tt >> 6], wa = cur0[tt >> 6];
        const int pb = (int)((wp >> (tt & 63)) & 1ull);
        const uint64_t pm = __ballot(pb);
        const uint64_t am = regular ? ~0ull : __ballot((int)((wa >> (tt & 63)) & 1ull));
        if (lane == 0) {
            S.par = pm;
            S.act = am;
        }
        if (CONS && lane < M::NB)
#pragma unroll
            for (int f = 0; f < 3; f++)
                S.shift[lane * 3 + f] = I.scal[8 + f] - I.s_tile[((int64_t)f * 2 + pb) * I.nt + tt];
    }
    __syncthreads();
    auto uniform = [](uint64_t w) {
        return ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(w >> 32)) << 32) |
               (uint32_t)__builtin_amdgcn_readfirstlane((int)w);
    };
    const uint64_t par = uniform(S.par), act = uniform(S.act);
    const int bw = min(M::TX, nx - x0) / 4, bh = min(M::TY, ny - y0) / 4;
    uint64_t own = 0ull;
    for (int j = 0; j < bh; j++) own |= ((1ull << bw) - 1ull) << (M::BW * (j + 1) + 1);
    if ((act & own) == 0ull) return;

    auto planes = [&](int f, gdouble*& b0, gdouble*& b1) {  // (as in the march)
        b0 = I.buf[0][f];
        b1 = I.buf[1][f];
        asm volatile("" : "+s"(b0), "+s"(b1));
    };
    // x, y, z of the region
    const bool two = tid >= M::NT - 64;
    double v[2][3];
    int lbit[2];
#pragma unroll
    for (int s = 0; s < 2; s++) {
        const int k = s == 0 ? tid : M::NT + lane, lx = k % M::CW, ly = k / M::CW;
        lbit[s] = ((lx + 2) >> 2) + M::BW * ((ly + 2) >> 2);
        const unsigned off = (unsigned)(wrap_any(x0 + lx - 2, nx) + wrap_any(y0 + ly - 2, ny) * nx) * 8u;
        const bool q = (par >> lbit[s]) & 1ull;
#pragma unroll
        for (int f = 0; f < 3; f++) {
            gdouble *b0, *b1;
            planes(f, b0, b1);
            v[s][f] = s == 0 || two ? at_bytes(q ? b1 : b0, off) : 0.0;
        }
    }
    // this thread's cell in the region of the potentials: a cell of the column, or of its ring
    int mx, my;
    if (tid < M::NI) {
        mx = 1 + (tid & 31);
        my = 1 + (tid >> 5);
    } else {
        const int r = min(tid - M::NI, M::NR - 1);
        if (r < 2 * M::MW) {
            mx = r < M::MW ? r : r - M::MW;
            my = r < M::MW ? 0 : M::MH - 1;
        } else {
            const int k = r - 2 * M::MW;
            mx = k < M::TY ? 0 : M::MW - 1;
            my = 1 + (k < M::TY ? k : k - M::TY);
        }
    }
    const bool cell = tid < M::NI;
    const bool mine = cell && mx - 1 < nx - x0 && my - 1 < ny - y0;  // a cell of the grid this column owns
    const int mbit = ((mx + 3) >> 2) + M::BW * ((my + 3) >> 2);
    const unsigned moff = (unsigned)(wrap_any(x0 + mx - 1, nx) + wrap_any(y0 + my - 1, ny) * nx) * 8u;
    const bool wakes = (act >> mbit) & 1ull, odd = (par >> mbit) & 1ull;
    double df[3], lap[3], phi;
    {
        gdouble *b0, *b1;
        planes(3, b0, b1);
        phi = at_bytes(odd ? b1 : b0, moff);
    }
    if (!wakes)
#pragma unroll
        for (int f = 0; f < 3; f++) df[f] = at_bytes(I.aux[f], moff);
#pragma unroll
    for (int f = 0; f < 3; f++) {
        if (CONS) {
            v[0][f] -= S.shift[lbit[0] * 3 + f];
            if (two) v[1][f] -= S.shift[lbit[1] * 3 + f];
        }
        S.c[f * M::CA + tid] = v[0][f];
        if (two) S.c[f * M::CA + M::NT + lane] = v[1][f];
    }
    __syncthreads();

    // the potentials
    double c[3];
#pragma unroll
    for (int f = 0; f < 3; f++) {
        const Plane3 n = plane_sums<M::CW>(S.c + (mx + 1) + (my + 1) * M::CW + f * M::CA);
        lap[f] = ((n.own + n.side) + n.side) * inv_dx2;
        c[f] = n.c;
    }
    if (wakes) {
        const double X = c[0], Y = c[1], Z = c[2], B = 1.0 - X - Y - Z;
        const double com = mb_shared(I, X, Y, Z, log_f64(B));
        __builtin_amdgcn_sched_barrier(0);
        df[0] = mb_mu_x<false>(I, Y, Z, B, com, log_f64(X), lap[0]);
        __builtin_amdgcn_sched_barrier(0);
        df[1] = mb_mu_y<false>(I, X, Z, B, com, log_f64(Y), lap[1]);
        __builtin_amdgcn_sched_barrier(0);
        df[2] = mb_mu_z<false>(I, X, Y, B, com, log_f64(Z), lap[2], phi);
        __builtin_amdgcn_sched_barrier(0);
    }
    double* sm = S.mu + mx + my * M::MW;
    if (tid < M::NI + M::NR)
#pragma unroll
        for (int f = 0; f < 3; f++) sm[f * M::MA] = df[f];
    if (cell && !regular) {
        const uint64_t w = __ballot(mine && wakes && fabs(lap[2]) > I.thresh_a);
        if (lane == 0) S.vote[wid] = w;
    }
    __syncthreads();
    if (cell) {
        const bool ran = mine && wakes;
        if (!regular && ran) {
            // the block's cells: four lanes in two rows, of this wave and its partner
            const uint64_t w = S.vote[wid & ~1] | S.vote[wid | 1];
            const bool fired = (w & ((0xFull | 0xFull << 32) << (tid & 28))) != 0ull;
            if (!fired)
#pragma unroll
                for (int f = 0; f < 3; f++) at_bytes(I.aux[f], moff) = df[f];
            if ((tid & 3) == 0 && ((tid >> 5) & 3) == 0) I.nflag[0][block_at(mbit)] = (uint8_t)fired;
        }
        // the changes
#pragma unroll
        for (int f = 0; f < 3; f++) {
            const Plane3 n = plane_sums<M::MW>(sm + f * M::MA);
            lap[f] = ((n.own + n.side) + n.side) * inv_dx2;
        }
        double ch[3];
        mb_change(I, df[0], df[1], df[2], lap[0], lap[1], lap[2], ch);
        if (ran)
#pragma unroll
            for (int f = 0; f < 3; f++) {
                gdouble *b0, *b1;
                planes(f, b0, b1);
                at_bytes(odd ? b0 : b1, moff) = c[f] + ch[f];
            }
        if (CONS)
#pragma unroll
            for (int f = 0; f < 3; f++) {
                double s = ran ? ch[f] : 0.0;
                s += __shfl_xor(s, 1, 64);
                s += __shfl_xor(s, 2, 64);
                s += __shfl_xor(s, 32, 64);
                if ((lane & 35) == 0) S.part[(f * (M::NI / 64) + wid) * 8 + (lane >> 2)] = s;
            }
    }
    if (CONS) {
        __syncthreads();
        // a block's change sums: its two waves' halves
        if (tid < 3 * (M::TY / 4) * 8) {
            const int f = tid / (8 * (M::TY / 4)), r = tid % (8 * (M::TY / 4)), j = r / 8, i = r % 8;
            const int bit = (i + 1) + M::BW * (j + 1);
            if (i < bw && j < bh && ((act >> bit) & 1ull)) {
                const int t = block_at(bit), b = (int)((par >> bit) & 1ull);
                const double* h = S.part + (f * (M::NI / 64) + 2 * j) * 8 + i;
                I.tpart[(int64_t)f * I.nt + t] = h[0] + h[8];
                I.s_tile[((int64_t)f * 2 + (b ^ 1)) * I.nt + t] = I.scal[8 + f];
            }
        }
    }
}

// ------------------------------------------------------------ Kobayashi-94 dendrite
//
// A wave per block, kK94Waves of them in a workgroup, each with its own part of the
// worklist and of LDS and no barrier between them. Lists are short here (a few
// thousand blocks), so a step is bound by the chain list entry -> bitmap words ->
// cells and by the dispatch of its workgroups, a long one by the instructions per
// block: the block's place, the parities of its six neighbours and the buffer choices
// are scalar (blocks divide the grid, so a face wraps as a whole), a lane's four
// loads per field differ by offsets, and the step's constants come from the host.
// 256^3 dendrite, one block per workgroup with a 27-neighbour table in LDS and per-cell
// index arithmetic -> this: 16.2 -> 11.1 us per launch over 2000 steps, 437 -> 335 us
// with all 262144 blocks awake.
constexpr int kK94Waves = 4;

template <int TB, int TZ>
__global__ __launch_bounds__(64 * kK94Waves) void k94_step_kernel(const WorkList wl) {
    static_assert(TB * TB * TZ <= 64, "a block is at most a wave");
    constexpr int WX = TB + 2, WZ = TZ + 2, A = WX * WX * WZ;
    __shared__ double box[kK94Waves][2][A];
    __shared__ FoldLds FL;
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    WorkCursor cur;
    // (the waves of one workgroup take neighbouring entries of its XCD's range)
    work_begin(wl, cur, false, ((int)(blockIdx.x >> 3) * kK94Waves + wid) * 8 + (int)(blockIdx.x & 7),
               (int)gridDim.x * kK94Waves);
    Fold FO;
    const int total = work_open(wl, FO, &FL);
    const int lx = lane % TB, ly = (lane / TB) % TB, lz = lane / (TB * TB);
    const bool mine = lane < TB * TB * TZ;
    const int q = (lx + 1) + (ly + 1) * WX + (mine ? lz + 1 : 1) * WX * WX;
    // where the lane's face cells go; a lane inside writes its own cell once more
    // (side: bit of the parities its face cell's block has)
    const int sx = lx == 0 ? 1 : (lx == TB - 1 ? 2 : 0), sy = ly == 0 ? 3 : (ly == TB - 1 ? 4 : 0);
    const int sz = lz == 0 ? 5 : (lz == TZ - 1 ? 6 : 0);
    const int qx = q + (sx == 1 ? -1 : (sx == 2 ? 1 : 0));
    const int qy = q + (sy == 3 ? -WX : (sy == 4 ? WX : 0));
    const int qz = q + (sz == 5 ? -WX * WX : (sz == 6 ? WX * WX : 0));
    double *sp = box[wid][0], *sT = box[wid][1];
    for (;;) {
        CInst* Ip;
        int t;
        uint64_t rec;
        if (!work_next(wl, FO, cur, total, &Ip, &t, &rec, false)) break;
        CInst& I = *Ip;
        const int nx = I.nx, ny = I.ny, ntx = I.ntx, nty = I.nty, ntz = I.ntz;
        const bool regular = I.mode == 0;
        gdouble *bp0 = I.buf[0][0], *bp1 = I.buf[1][0], *bT0 = I.buf[0][1], *bT1 = I.buf[1][1];
        const DBA_CONST uint64_t *par0 = (const DBA_CONST uint64_t*)I.par[0], *par1 = (const DBA_CONST uint64_t*)I.par[1];
        const DBA_CONST uint64_t *act0 = (const DBA_CONST uint64_t*)I.a_cur[0], *act1 = (const DBA_CONST uint64_t*)I.a_cur[1];
        const double f0 = I.k94_f0, f1 = I.k94_f1, f2 = I.k94_f2, f3 = I.k94_f3;
        const double dt = I.dt, eps = I.eps_bar, delta = I.delta, gam = I.gamma;
        asm volatile("" : "+s"(bp0), "+s"(bp1), "+s"(bT0), "+s"(bT1));
        const int tt = t / ntx, ti = t - tt * ntx, tk = TZ == 1 ? 0 : tt / nty, tj = tt - tk * nty;
        const int xm = ti > 0 ? ti - 1 : ntx - 1, xp = ti < ntx - 1 ? ti + 1 : 0;
        const int ym = tj > 0 ? tj - 1 : nty - 1, yp = tj < nty - 1 ? tj + 1 : 0;
        const int zm = tk > 0 ? tk - 1 : ntz - 1, zp = tk < ntz - 1 ? tk + 1 : 0;
        const int n_xm = t + xm - ti, n_xp = t + xp - ti, n_ym = t + (ym - tj) * ntx, n_yp = t + (yp - tj) * ntx;
        const int n_zm = t + (zm - tk) * ntx * nty, n_zp = t + (zp - tk) * ntx * nty;
        auto bit = [](const DBA_CONST uint64_t* m, int k) { return (uint32_t)(m[k >> 6] >> (k & 63)) & 1u; };
        // parities of the block (bit 0) and of its neighbours below and above in x, y, z
        auto parities = [&](const DBA_CONST uint64_t* m) {
            return bit(m, t) | bit(m, n_xm) << 1 | bit(m, n_xp) << 2 | bit(m, n_ym) << 3 | bit(m, n_yp) << 4 |
                   bit(m, n_zm) << 5 | bit(m, n_zp) << 6;
        };
        const uint32_t ap = regular ? 1u : bit(act0, t), at = regular ? 1u : bit(act1, t);
        const uint32_t pp = parities(par0), pT = parities(par1);

        // the lane's cell, and from it to its face cells (0: not on that face)
        const int64_t nxy = (int64_t)nx * ny;
        const int x = ti * TB + lx, y = tj * TB + ly, z = tk * TZ + (mine ? lz : 0);
        const int64_t own = x + (int64_t)y * nx + z * nxy;
        const int fx = sx == 1 ? xm * TB + TB - 1 - x : (sx == 2 ? xp * TB - x : 0);
        const int fy = sy == 3 ? ym * TB + TB - 1 - y : (sy == 4 ? yp * TB - y : 0);
        const int fz = TZ == 1 ? 0 : (sz == 5 ? zm * TZ + TZ - 1 - z : (sz == 6 ? zp * TZ - z : 0));
        const int64_t ox = own + fx, oy = own + (int64_t)fy * nx, oz = own + fz * nxy;
        auto from = [](const gdouble* b0, const gdouble* b1, uint32_t par, int side, int64_t o) {
            return ((par >> side) & 1u ? b1 : b0)[o];
        };
        double vpx = 0.0, vpy = 0.0, vpz = 0.0, vTx = 0.0, vTy = 0.0, vTz = 0.0;
        const double vp = ((pp & 1u) ? bp1 : bp0)[own];
        const double vT = ((pT & 1u) ? bT1 : bT0)[own];
        if (ap) {
            vpx = from(bp0, bp1, pp, sx, ox);
            vpy = from(bp0, bp1, pp, sy, oy);
            if (TZ > 1) vpz = from(bp0, bp1, pp, sz, oz);
        }
        if (at) {
            vTx = from(bT0, bT1, pT, sx, ox);
            vTy = from(bT0, bT1, pT, sy, oy);
            if (TZ > 1) vTz = from(bT0, bT1, pT, sz, oz);
        }
        if (mine) {
            sp[q] = vp;
            sT[q] = vT;
            if (ap) {
                sp[qx] = vpx;
                sp[qy] = vpy;
                if (TZ > 1) sp[qz] = vpz;
                else sp[q - WX * WX] = sp[q + WX * WX] = vp;  // one plane: its own neighbour
            }
            if (at) {
                sT[qx] = vTx;
                sT[qy] = vTy;
                if (TZ > 1) sT[qz] = vTz;
                else sT[q - WX * WX] = sT[q + WX * WX] = vT;
            }
        }
        wave_lds_sync();
        int fp = 0, fT = 0;
        if (mine) {
            const double pc = vp, Tc = vT;
            double pn = pc;
            if (ap) {
                const double pxp_ = sp[q + 1], pxm_ = sp[q - 1], pyp_ = sp[q + WX], pym_ = sp[q - WX];
                const double pzp_ = sp[q + WX * WX], pzm_ = sp[q - WX * WX];
                const double dpx = (pxp_ - pxm_) * f0, dpy = (pyp_ - pym_) * f0, dpz = (pzp_ - pzm_) * f0;
                const double lapP = (pxp_ + pxm_ + pyp_ + pym_ + pzp_ + pzm_ - 6 * pc) * f1;
                const double v2 = dpx * dpx + dpy * dpy + dpz * dpz;
                double sigma;
                if (v2 <= 1E-6)
                    sigma = 1;
                else
                    sigma = 1 - delta * (1 - ((dpx * dpx) * (dpx * dpx) + (dpy * dpy) * (dpy * dpy) +
                                              (dpz * dpz) * (dpz * dpz)) / (v2 * v2));
                const double m = f2 * atan(gam * sigma * Tc);
                const double p_change = f3 * (eps * eps * lapP + pc * (1 - pc) * (pc - 0.5 + m));
                pn = pc + dt * p_change;
                ((pp & 1u) ? bp0 : bp1)[own] = pn;
                fp = pn >= I.thresh_a && pn <= (1.0 - I.thresh_a);
            }
            if (at) {
                const double lapT = (sT[q + 1] + sT[q - 1] + sT[q + WX] + sT[q - WX] + sT[q + WX * WX] +
                                     sT[q - WX * WX] - 6 * Tc) * f1;
                double tn;
                if (regular) {
                    tn = Tc + dt * lapT + pn - pc;
                } else {
                    tn = Tc + dt * lapT;
                    if (ap) tn += pn - pc;
                }
                ((pT & 1u) ? bT0 : bT1)[own] = tn;
                fT = fabs(tn - Tc) >= I.thresh_b;
            }
        }
        if (!regular) {
            const int anyp = __ballot(fp) != 0ull, anyT = __ballot(fT) != 0ull;
            if (lane == 0) {
                if (ap) I.nflag[0][t] = (uint8_t)anyp;
                if (at) I.nflag[1][t] = (uint8_t)anyT;
            }
        }
        wave_lds_sync();  // the next block's cells come after this one's reads
    }
}

}  // namespace dba
