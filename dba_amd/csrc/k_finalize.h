// k_finalize.h - end-of-step activation bookkeeping and worklist compaction.
//
// Reference counterpart: the tail of every DBA step, Wakeup_Next (clears the
// flags of the blocks that ran, example_Dendritic_growth/kernel.cu:496-574)
// and Wakeup_Neighbor (sets each flagged block and its neighbours,
// kernel.cu:577-634; 3x3 in KH, example_Kelvin_Helmholtz/KH_DBA.cu:988-1044),
// plus the conserved mean shift (example_Reactive_ModelB/Conserved/kernel.cu:1152-1164).
//
// One workgroup per segment of <= 1024 tiles:
//   (a) counts the tiles that ran (history), flips their buffer parity, and
//       sums their conserved change partials;
//   (b) dilates the detector bytes of the step into the next awake set: each
//       lane evaluates one tile, a wave ballot gives a 64-tile bitmap word;
//   (c) compacts the segment's union awake set into an ascending list
//       (popcount prefix over the segment's words, then the lane's rank in
//       its word), i.e. the order copy_if over tile indices gives;
//   (d) of a one-segment group, updates the instance (history, counters, conserved
//       shift, KH CFL dt); of several segments it leaves partial sums and counts,
//       which a merge launch sums per instance in segment order and scans into the
//       list's offsets, or, where no step needs the sums of the one before, which the
//       next step's kernel scans and the next finalize sums (folded merges, common.h).
#pragma once
#include "common.h"

namespace dba {

__device__ __forceinline__ uint64_t full_word(int w, int nt) {
    int n = nt - w * 64;
    if (n >= 64) return ~0ull;
    if (n <= 0) return 0ull;
    return (1ull << n) - 1ull;
}

__device__ __forceinline__ int64_t tile_cells(CInst& I, int t) {
    int ti = t % I.ntx, tj = (t / I.ntx) % I.nty, tk = t / (I.ntx * I.nty);
    int wx = min(I.tx, I.nx - ti * I.tx), wy = min(I.ty, I.ny - tj * I.ty), wz = min(I.tz, I.nz - tk * I.tz);
    return (int64_t)wx * wy * wz;
}

// 2D tile grid: neighbour columns/rows resolved once (-1 = clamped away).
struct Nb2 {
    int xm, xp, ym, yp;  // tile-grid column / row indices
};

__device__ __forceinline__ Nb2 nb2_of(int ti, int tj, int ntx, int nty, int bcx, int bcy) {
    Nb2 n;
    n.xm = ti > 0 ? ti - 1 : (bcx == 0 ? ntx - 1 : -1);
    n.xp = ti < ntx - 1 ? ti + 1 : (bcx == 0 ? 0 : -1);
    n.ym = tj > 0 ? tj - 1 : (bcy == 0 ? nty - 1 : -1);
    n.yp = tj < nty - 1 ? tj + 1 : (bcy == 0 ? 0 : -1);
    return n;
}

// Awake flag of tile (ti, tj) for the next step (CH, K93): OR of the detector bytes
// over the tile and its face neighbours.
__device__ __forceinline__ int dilated2d(const gu8* N, int ti, int tj, int ntx, const Nb2& n) {
    // A missing neighbour (zero-flux boundary) reads the tile itself instead, which
    // the OR already holds: no load depends on a branch, so all of them are in flight
    // at once instead of one after another.
    const int xm = n.xm >= 0 ? n.xm : ti, xp = n.xp >= 0 ? n.xp : ti;
    const int ym = n.ym >= 0 ? n.ym : tj, yp = n.yp >= 0 ? n.yp : tj;
    const int row = tj * ntx, rm = ym * ntx, rp = yp * ntx;
    return (N[ti + row] | N[xm + row] | N[xp + row] | N[ti + rm] | N[ti + rp]) != 0;
}

template <int NT>
__device__ __forceinline__ int block_exclusive_scan(int v, int* lds, int* total) {
    constexpr int NW = NT / 64;
    int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    int incl = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        int y = __shfl_up(incl, off, 64);
        if (lane >= off) incl += y;
    }
    if (lane == 63) lds[wid] = incl;
    __syncthreads();
    int base = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < NW; w++) {
        int c = lds[w];
        if (w < wid) base += c;
        tot += c;
    }
    __syncthreads();
    *total = tot;
    return base + incl - v;
}

constexpr int kFinNT = 1024;  // one tile per thread for a full segment
constexpr int kSegWords = kSegTiles / 64;

// Per-instance end-of-step update from the summed segment partials.
__device__ __forceinline__ void finish_instance(CInst& J, int64_t listlen, unsigned long long c0,
                                                unsigned long long c1, unsigned long long cells, const double* cs,
                                                double vmax, int64_t step, int64_t updates, const double* scal_in,
                                                int rotate) {
    J.ctr[2] = listlen;
    if (!rotate) return;
    if (step < J.hist_cap) {
        J.hist[2 * step] = (int32_t)c0;
        J.hist[2 * step + 1] = J.nsets > 1 ? (int32_t)c1 : 0;
    }
    J.ctr[0] = step + 1;
    J.ctr[1] = updates + (int64_t)cells;
    for (int f = 0; f < J.ncons; f++) J.scal[8 + f] = scal_in[8 + f] + cs[f] / J.ntotal;
    const double used = scal_in[1];
    J.scal[2] = scal_in[2] + used;
    J.scal[3] = used;
    if (J.model == 5 && J.dt_mode == 1) J.scal[1] = J.cfl * (J.dx / vmax);
}

// Merge of one instance's segment partials (segments [first, first + count)) by
// one wave: lanes stride over the segments, then a fixed-shape shuffle tree (the
// same order on every run, and for a one-segment instance exactly that segment's
// partial). counts: null leaves the list length as it is.
__device__ __forceinline__ void merge_instance(CInst& J, int first, int count, const SegPart* __restrict__ parts,
                                               const int32_t* __restrict__ counts, int rotate) {
    const int lane = threadIdx.x & 63;
    // the descriptor's fields in one batch, then the instance's scalars and counters
    // with the partials: no load waits for another
    const int ncs = J.ncons, model = J.model, dt_mode = J.dt_mode, nsets = J.nsets, hist_cap = J.hist_cap;
    gdouble* scal = J.scal;
    gi64* ctr = J.ctr;
    gi32* hist = J.hist;
    const double ntotal = J.ntotal, cfl_n = J.cfl, dx = J.dx;
    asm volatile("" ::"s"(ncs), "s"(model), "s"(dt_mode), "s"(nsets), "s"(hist_cap), "s"(scal), "s"(ctr), "s"(hist),
                 "s"(ntotal), "s"(cfl_n), "s"(dx));
    const bool cfl = rotate && model == 5 && dt_mode == 1;
    double sc[16] = {0.0};
    sc[1] = scal[1];
    sc[2] = scal[2];
#pragma unroll
    for (int f = 0; f < kMaxFields; f++) sc[8 + f] = scal[8 + f];
    const int64_t step = ctr[0], upd = ctr[1], len = ctr[2];
    int ll = 0;
    unsigned long long q01 = 0, qc = 0;  // tiles that ran set 0, set 1 << 32; their cells
    double cs[kMaxFields] = {0.0, 0.0, 0.0, 0.0};
    double vm = 0.0;
#pragma unroll 2
    for (int q = first + lane; q < first + count; q += 64) {
        if (counts) ll += counts[q];
        if (rotate) {
            q01 += parts[q].c0 | parts[q].c1 << 32;
            qc += parts[q].cells;
#pragma unroll
            for (int f = 0; f < kMaxFields; f++)
                if (f < ncs) cs[f] += parts[q].csum[f];
            if (cfl) vm = fmax(vm, parts[q].vmax);
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        ll += __shfl_down(ll, off, 64);
        q01 += __shfl_down(q01, off, 64);
        qc += __shfl_down(qc, off, 64);
    }
#pragma unroll
    for (int f = 0; f < kMaxFields; f++)
        if (f < ncs) cs[f] = wave_sum_down(cs[f]);
    if (cfl) vm = wave_max_down(vm);
    if (lane == 0)
        finish_instance(J, counts ? (int64_t)ll : len, q01 & 0xffffffffull, q01 >> 32, qc, cs, vm, step, upd, sc, rotate);
}

// LDS of the finalize body.
struct FinLds {
    uint8_t bits[kSegTiles];        // per tile: awake in the next step (bits 0, 1: sets), parity it sees (2, 3)
    alignas(16) int listed[kSegWords];  // per 64-tile word: tiles in the next worklist
    alignas(16) uint32_t ran[kSegWords];    // ... tiles that ran: set 0, set 1 << 16
    alignas(16) uint32_t cells[kSegWords];  // ... and their cells
    double csum[kMaxFields][kSegWords];     // ... conserved change sums
    double vmax[kSegWords];                 // ... KH wave speed
};

// One thread per tile of the segment, one wave per 64-tile bitmap word, one
// workgroup barrier.
//
// What bounds it: the chain of dependent loads (a segment has 30 KB of state). The
// descriptor's fields come in one batch of scalar loads, then every vector load of
// both sets goes out before the first is waited for; past the barrier everything is
// read from LDS at fixed addresses, and folded merges have a workgroup of their own.
// With loads waited for branch by branch and LDS loops of the segment's length, us per
// launch before -> now: 16 dendrites in 30 segments 8.5 -> 5.4, a 256^3 dendrite (256
// segments) 7.7 -> 5.8, KH 2048^2 (16 segments) 7.9 -> 5.3, 96 x 80 x 64
// conserved Model B 7.3 -> 5.0.
template <int NT>
__device__ __forceinline__ void finalize_body(const Inst* __restrict__ insts, const Seg* __restrict__ segs,
                                              int segi, int nseg, SegPart* __restrict__ parts,
                                              int32_t* __restrict__ counts, int32_t* __restrict__ offsets,
                                              int rotate, int one_inst, FinLds& F) {
    static_assert(NT == kSegTiles, "one thread per tile of a segment");
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    // one segment: instance 0, all of its tiles (no dependent load of the segment table)
    // one instance: segment segi holds its tiles from segi kSegTiles on, so the
    // segment table is not read (its load would come before the descriptor's)
    const bool solo = nseg == 1, one = solo || one_inst;
    int inst = 0, t0 = solo ? 0 : segi * kSegTiles, seg_n = 0;
    if (!one) {
        const Seg sg = segs[segi];
        inst = __builtin_amdgcn_readfirstlane(sg.inst);
        t0 = __builtin_amdgcn_readfirstlane(sg.tile0);
        seg_n = __builtin_amdgcn_readfirstlane(sg.ntile);
    }
    CInst& I = ((CInst*)insts)[inst];
    const int nt = I.nt, ntx = I.ntx, nty = I.nty, ntz = I.ntz, bcx = I.bc_x, bcy = I.bc_y, bcz = I.bc_z;
    const int mode = I.mode, nsets = I.nsets, model = I.model, ncons = I.ncons, dt_mode = I.dt_mode;
    const int tile_n = I.tx * I.ty * I.tz, full_tiles = I.full_tiles;
    gu64 *cur0p = I.a_cur[0], *cur1p = I.a_cur[1], *par0p = I.par[0], *par1p = I.par[1];
    const gu8 *nf0 = I.nflag[0], *nf1 = I.nflag[1];
    const gdouble *tpart = I.tpart, *tspeed = I.tspeed;
    gi32* seg = I.seg;
    gu64* nbrec = I.nbrec;
    asm volatile("" ::"s"(nt), "s"(ntx), "s"(nty), "s"(ntz), "s"(bcx), "s"(bcy), "s"(bcz), "s"(mode), "s"(nsets),
                 "s"(model), "s"(ncons), "s"(dt_mode), "s"(tile_n), "s"(full_tiles), "s"(cur0p), "s"(cur1p),
                 "s"(par0p), "s"(par1p), "s"(nf0), "s"(nf1), "s"(tpart), "s"(tspeed), "s"(seg), "s"(nbrec));
    const int nts = solo ? nt : (one_inst ? min(kSegTiles, nt - t0) : seg_n);
    const int w0 = t0 >> 6, nws = (nts + 63) >> 6;
    const bool regular = mode == 0, dilate = rotate && !regular, cfl = rotate && model == 5 && dt_mode == 1;
    const int t = t0 + tid, tc = tid < nts ? t : t0;
    const bool valid = tid < nts;
    const bool wvalid = wid < nws;  // this wave's word exists

    // ---- every global load, issued together (past the segment: tile t0's, not used)
    const int wc = w0 + (wvalid ? wid : 0);
    uint64_t cur0 = regular ? full_word(wc, nt) : cur0p[wc], par0 = par0p[wc], cur1 = 0ull, par1 = 0ull;
    if (nsets > 1) {
        cur1 = regular ? full_word(wc, nt) : cur1p[wc];
        par1 = par1p[wc];
    }
    const int q = tc / ntx, ti = tc - q * ntx, tk = ntz == 1 ? 0 : q / nty, tj = q - tk * nty;
    // neighbour columns, rows and planes; one clamped away is the tile's own
    const int xm = ti > 0 ? ti - 1 : (bcx == 0 ? ntx - 1 : ti), xp = ti < ntx - 1 ? ti + 1 : (bcx == 0 ? 0 : ti);
    const int ym = tj > 0 ? tj - 1 : (bcy == 0 ? nty - 1 : tj), yp = tj < nty - 1 ? tj + 1 : (bcy == 0 ? 0 : tj);
    int f0[11], f1[7];
#pragma unroll
    for (int k = 0; k < 11; k++) f0[k] = 0;
#pragma unroll
    for (int k = 0; k < 7; k++) f1[k] = 0;
    if (dilate) {
        const int nxy = ntx * nty, pl = tk * nxy, row = tj * ntx + pl, rm = ym * ntx + pl, rp = yp * ntx + pl;
        const int o[5] = {tc, xm + row, xp + row, ti + rm, ti + rp};
        const int zm = tk > 0 ? tk - 1 : (bcz == 0 ? ntz - 1 : tk), zp = tk < ntz - 1 ? tk + 1 : (bcz == 0 ? 0 : tk);
        const int om = zm * nxy + tj * ntx + ti, op = zp * nxy + tj * ntx + ti;
#pragma unroll
        for (int k = 0; k < 5; k++) f0[k] = nf0[o[k]];
        if (ntz > 1) {
            f0[5] = nf0[om];
            f0[6] = nf0[op];
        }
        if (model == 5) {  // 3x3 in the plane
            f0[7] = nf0[xm + rm];
            f0[8] = nf0[xp + rm];
            f0[9] = nf0[xm + rp];
            f0[10] = nf0[xp + rp];
        }
        if (nsets > 1) {
#pragma unroll
            for (int k = 0; k < 5; k++) f1[k] = nf1[o[k]];
            if (ntz > 1) {
                f1[5] = nf1[om];
                f1[6] = nf1[op];
            }
        }
    }
    double part[kMaxFields] = {0.0, 0.0, 0.0, 0.0};
    if (rotate)
#pragma unroll
        for (int f = 0; f < kMaxFields; f++)
            if (f < ncons) part[f] = tpart[(int64_t)f * nt + tc];
    double fresh = 0.0, stale = 0.0;
    if (cfl) {
        fresh = tspeed[tc];
        stale = tspeed[nt + tc];
    }

    double sc[16] = {0.0};
    int64_t step = 0, upd = 0;
    if (solo) {  // what finish_instance needs
        sc[1] = I.scal[1];
        sc[2] = I.scal[2];
#pragma unroll
        for (int f = 0; f < kMaxFields; f++) sc[8 + f] = I.scal[8 + f];
        step = I.ctr[0];
        upd = I.ctr[1];
    }

    // ---- this tile: ran in the executed step?  awake in the next?  parity next?
    if (!wvalid) cur0 = cur1 = par0 = par1 = 0ull;
    const int ran0 = (int)((cur0 >> lane) & 1ull), ran1 = (int)((cur1 >> lane) & 1ull);
    int b0 = ran0, b1 = ran1;  // regular: every tile every step; rebuild (rotate = 0): the current sets
    if (dilate) {
        b0 = (f0[0] | f0[1] | f0[2] | f0[3] | f0[4] | f0[5] | f0[6] | f0[7] | f0[8] | f0[9] | f0[10]) != 0;
        b1 = (f1[0] | f1[1] | f1[2] | f1[3] | f1[4] | f1[5] | f1[6]) != 0;
    }
    if (!valid) b0 = b1 = 0;
    const uint64_t pn0 = rotate ? (par0 ^ cur0) : par0;
    const uint64_t pn1 = rotate ? (par1 ^ cur1) : par1;
    const uint64_t nw0 = __ballot(b0);
    const uint64_t nw1 = __ballot(b1);
    const uint64_t uni = nw0 | nw1;
    F.bits[tid] = (uint8_t)(b0 | b1 << 1 | (int)((pn0 >> lane) & 1ull) << 2 | (int)((pn1 >> lane) & 1ull) << 3);
    if (rotate && wvalid && lane == 0) {
        par0p[w0 + wid] = pn0;
        if (nsets > 1) par1p[w0 + wid] = pn1;
        if (!regular) {
            cur0p[w0 + wid] = nw0;
            if (nsets > 1) cur1p[w0 + wid] = nw1;
        }
    }
    // per-word statistics of the executed step
    // field-set updates: set 0's fields over the tiles that ran it; the second
    // set's field (dendrite T) over the tiles that ran either set, since a
    // p-awake tile writes T too
    uint32_t cells = 0;
    if (rotate) {
        if (full_tiles) {
            cells = (uint32_t)tile_n * (uint32_t)(__popcll(cur0 | cur1) + (nsets > 1 ? __popcll(cur0) : 0));
        } else {
            if (valid && (ran0 | ran1)) cells = (uint32_t)tile_cells(I, t) * (uint32_t)(nsets > 1 ? 1 + ran0 : 1);
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) cells += __shfl_down(cells, off, 64);
        }
    }
    if (lane == 0) {
        F.listed[wid] = __popcll(uni);
        F.ran[wid] = (uint32_t)__popcll(cur0) | (uint32_t)__popcll(cur1) << 16;
        F.cells[wid] = cells;
    }
    // conserved change sums of the tiles that ran (sleeping tiles contribute 0):
    // block_sum's tree, its words added in order below
    if (rotate)
#pragma unroll
        for (int f = 0; f < kMaxFields; f++)
            if (f < ncons) {
                const double s = wave_sum_down(valid && ran0 ? part[f] : 0.0);
                if (lane == 0) F.csum[f][wid] = s;
            }
    // KH: max wave speed the next step's CFL sees (fresh for awake tiles, stale otherwise)
    if (cfl) {
        const double v = wave_max_down(valid ? (b0 ? fresh : stale) : 0.0);
        if (lane == 0) F.vmax[wid] = v;
    }
    __syncthreads();

    // ---- compaction of the union set (ascending tiles) and the neighbour records
    int base = 0, listlen = 0;
#pragma unroll
    for (int w = 0; w < kSegWords; w++) {
        const int c = F.listed[w];
        if (w < wid) base += c;
        listlen += c;
    }
    if ((uni >> lane) & 1ull) {
        const int pos = t0 + base + __popcll(uni & ((1ull << lane) - 1ull));
        seg[pos] = t;
        if (ntz == 1) {
            // resolved here when all nine owners are in this segment
            uint64_t rec = kRecValid;
            bool all = true;
#pragma unroll
            for (int d = 0; d < 9; d++) {
                const int o = (d % 3 == 0 ? xm : (d % 3 == 1 ? ti : xp)) +
                              (d / 3 == 0 ? ym : (d / 3 == 1 ? tj : yp)) * ntx - t0;
                const bool here = o >= 0 && o < nts;
                all = all && here;
                const uint32_t v = F.bits[here ? o : 0];
                rec |= (uint64_t)((v >> 2) & 1u) << d | (uint64_t)(v & 1u) << (9 + d) |
                       (uint64_t)(v >> 3) << (18 + d) | (uint64_t)((v >> 1) & 1u) << (27 + d);
            }
            nbrec[pos] = all ? rec : 0ull;
        }
    }
    if (tid != 0) return;

    // ---- the segment's sums
    uint32_t ran = 0, ncell = 0;
#pragma unroll
    for (int w = 0; w < kSegWords; w++) {
        ran += F.ran[w];  // (at most 1024 of each set: no carry)
        ncell += F.cells[w];
    }
    double cs[kMaxFields] = {0.0, 0.0, 0.0, 0.0};
    if (rotate)
#pragma unroll
        for (int f = 0; f < kMaxFields; f++)
            if (f < ncons)
                for (int w = 0; w < kSegWords; w++) cs[f] += F.csum[f][w];
    double vmax = 0.0;
    if (cfl) {
        vmax = F.vmax[0];
        for (int w = 1; w < kSegWords; w++) vmax = fmax(vmax, F.vmax[w]);
    }
    const unsigned long long c0 = ran & 0xffffu, c1 = ran >> 16;
    if (solo) {
        finish_instance(I, listlen, c0, c1, ncell, cs, vmax, step, upd, sc, rotate);
        offsets[0] = 0;
        offsets[1] = listlen;
        return;
    }
    counts[segi] = listlen;
    if (rotate) {
        parts[segi].c0 = c0;
        parts[segi].c1 = c1;
        parts[segi].cells = ncell;
        for (int f = 0; f < kMaxFields; f++) parts[segi].csum[f] = cs[f];
        parts[segi].vmax = vmax;
    }
}

// Several segments: one workgroup merges the segment partials after the
// segment workgroups (the kernel boundary makes their writes visible; a
// last-workgroup-done counter would need an agent-scope fence in every
// segment workgroup, and each such fence writes back and invalidates its XCD's
// L2). Per instance, one wave: lanes stride over the instance's segments, then a
// fixed-shape shuffle tree (the same order on every run, and for a one-segment
// instance exactly that segment's partial). Then the merged list offsets.
template <int NT>
__device__ __forceinline__ void finalize_merge_body(const Inst* __restrict__ insts, int nseg,
                                                    const InstSegs* __restrict__ isegs, int n_inst,
                                                    const SegPart* __restrict__ parts,
                                                    const int32_t* __restrict__ counts,
                                                    int32_t* __restrict__ offsets, int rotate, int* si) {
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    // One workgroup: the instances (a wave each, NT/64 at a time), then the
    // offsets scan. Several: workgroup 0 scans, workgroup b >= 1 takes
    // instances [(b-1) NT/64, b NT/64), all at once.
    const bool one = gridDim.x == 1;
    int i_lo = 0, i_hi = n_inst;  // this workgroup's instances
    if (!one) {
        i_lo = blockIdx.x == 0 ? 0 : ((int)blockIdx.x - 1) * (NT / 64);
        i_hi = blockIdx.x == 0 ? 0 : min(n_inst, i_lo + NT / 64);
    }
    // the offsets scan's first counts, loaded with the reductions' inputs
    const int v_first = tid < nseg ? counts[tid] : 0;
    for (int i0 = i_lo; i0 < i_hi; i0 += NT / 64) {
        const int i = i0 + wid;
        if (i >= i_hi) break;
        CInst& J = ((CInst*)insts)[i];
        const InstSegs r = n_inst == 1 ? InstSegs{0, nseg} : isegs[i];
        merge_instance(J, r.first, r.count, parts, counts, rotate);
    }
    if (!one && blockIdx.x != 0) return;
    int running = 0;
    for (int b = 0; b < nseg; b += NT) {
        const int i = b + tid;
        const int v = b == 0 ? v_first : (i < nseg ? counts[i] : 0);
        int tot;
        const int ex = block_exclusive_scan<NT>(v, si, &tot);
        if (i < nseg) offsets[i] = running + ex;
        running += tot;
    }
    if (tid == 0) offsets[nseg] = running;
}


// Workgroups past the segments (folded merges): the instance sums of the step
// before this one, a wave per instance.
__global__ __launch_bounds__(kFinNT) void finalize_kernel(const Inst* __restrict__ insts,
                                                          const Seg* __restrict__ segs, int nseg,
                                                          SegPart* __restrict__ parts,
                                                          int32_t* __restrict__ counts,
                                                          int32_t* __restrict__ offsets, int rotate,
                                                          int one_inst, const SegPart* __restrict__ pend,
                                                          const InstSegs* __restrict__ isegs, int n_inst) {
    __shared__ FinLds F;
    if ((int)blockIdx.x >= nseg) {
        const int i = ((int)blockIdx.x - nseg) * (kFinNT / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        if (i >= n_inst) return;
        const InstSegs r = n_inst == 1 ? InstSegs{0, nseg} : isegs[i];
        merge_instance(((CInst*)insts)[i], r.first, r.count, pend, nullptr, 1);
        return;
    }
    finalize_body<kFinNT>(insts, segs, blockIdx.x, nseg, parts, counts, offsets, rotate, one_inst, F);
}

__global__ __launch_bounds__(kFinNT) void finalize_merge_kernel(const Inst* __restrict__ insts, int nseg,
                                                                const InstSegs* __restrict__ isegs, int n_inst,
                                                                const SegPart* __restrict__ parts,
                                                                const int32_t* __restrict__ counts,
                                                                int32_t* __restrict__ offsets, int rotate) {
    __shared__ int si[kFinNT / 64 + 2];
    finalize_merge_body<kFinNT>(insts, nseg, isegs, n_inst, parts, counts, offsets, rotate, si);
}

// Instance and tile of a single-launch step's workgroup. With `deal`, workgroups
// are dealt to XCDs in contiguous ranges (the worklist kernels' deal), so halo
// rows a neighbour tile wrote last step are in this XCD's L2 (CH, every tile
// active); without, tile b goes to XCD b % 8, which spreads a sparse set of
// awake tiles over all XCDs (K93, whose awake tiles cluster in a few rows). A group of several
// instances or segments maps the dealt index through dmap (instance << 24 |
// tile, the instances' tiles in group order); one instance in one segment
// uses the index itself.
__device__ __forceinline__ CInst& dense_item(const Inst* insts, const int32_t* dmap, int* t, bool deal = true) {
    const int b = deal ? xcd_deal(blockIdx.x, gridDim.x, 0, gridDim.x) : (int)blockIdx.x;
    if (!dmap) {
        *t = b;
        return ((CInst*)insts)[0];
    }
    const uint32_t d = (uint32_t)dmap[b];
    *t = (int)(d & 0xFFFFFFu);
    return ((CInst*)insts)[d >> 24];
}

// The detector and parity bytes a single-launch step reads (step parity prev):
// the four arrays' pointers in one batch of scalar loads, then a select. The
// empty asm keeps the compiler from turning the select of two loaded pointers
// back into a load from a selected address, which put a dependent scalar load
// in front of each array's bytes.
__device__ __forceinline__ void dense_bytes(CInst& I, int prev, const gu8** F, const gu8** P) {
    const gu8* F0 = I.dF[0];
    const gu8* F1 = I.dF[1];
    const gu8* P0 = I.dP[0];
    const gu8* P1 = I.dP[1];
    asm volatile("" : "+s"(F0), "+s"(F1), "+s"(P0), "+s"(P1));
    *F = prev ? F1 : F0;
    *P = prev ? P1 : P0;
}

// The descriptor fields a single-launch step reads before its first barrier,
// as one batch of scalar loads at the start of the workgroup: the empty asm
// needs every value at that point, so the loads issue together and cost one
// round trip, where the compiler had placed them one dependent wait after another.
__device__ __forceinline__ void dense_prefetch(CInst& I, int nfield) {
    const int nt = I.nt, ntx = I.ntx, nty = I.nty, nx = I.nx, ny = I.ny, bcx = I.bc_x, bcy = I.bc_y, mode = I.mode;
    const gu8 *f0 = I.dF[0], *f1 = I.dF[1], *p0 = I.dP[0], *p1 = I.dP[1];
    const gi32* runs = I.druns;
    const gdouble *b00 = I.buf[0][0], *b10 = I.buf[1][0];
    const gdouble *b01 = nfield > 1 ? I.buf[0][1] : b00, *b11 = nfield > 1 ? I.buf[1][1] : b10;
    asm volatile("" ::"s"(nt), "s"(ntx), "s"(nty), "s"(nx), "s"(ny), "s"(bcx), "s"(bcy), "s"(mode), "s"(f0), "s"(f1),
                 "s"(p0), "s"(p1), "s"(runs), "s"(b00), "s"(b10), "s"(b01), "s"(b11));
}

// Neighbour table of a single-launch step (threads 0..8; caller synchronises):
// per set, buffer parity and awake bit of each 3x3 owner tile, from the bitmaps
// at the first step of a run, afterwards from the previous step's per-tile bytes
// (awake = the 5-point dilation of its detector bits, the finalize's rule).
// dF / dP hold, per step parity, nsets x nt bytes (set-major).
__device__ __forceinline__ void dense_nb_fill(NbTable& nb, CInst& I, int t, int first, int prev, bool regular,
                                              int nsets, bool cons) {
    const int d = threadIdx.x;
    if (d >= 9) return;
    const int nt = I.nt, ntx = I.ntx, tj = t / ntx, ti = t - tj * ntx;
    const int o = nb_owner2d(I, ti, tj, d);
    const int oj = o / ntx, oi = o - oj * ntx;
    nb.tile[d] = o;
    // every load first (both sets, the conserved epochs), then the table
    const double e0 = cons ? I.s_tile[o] : 0.0, e1 = cons ? I.s_tile[nt + o] : 0.0;
    int par[2] = {0, 0}, act[2] = {1, 1};
    if (first) {
        for (int s = 0; s < nsets; s++) par[s] = bit_of(I.par[s], o);
        if (!regular)
            for (int s = 0; s < nsets; s++) act[s] = bit_of(I.a_cur[s], o);
    } else {
        const Nb2 n = nb2_of(oi, oj, ntx, I.nty, I.bc_x, I.bc_y);
        const gu8 *F, *P;
        dense_bytes(I, prev, &F, &P);
        for (int s = 0; s < nsets; s++) par[s] = P[s * nt + o];
        if (!regular)
            for (int s = 0; s < nsets; s++) act[s] = dilated2d(F + s * nt, oi, oj, ntx, n);
    }
    for (int s = 0; s < nsets; s++) {
        nb.par[s][d] = par[s];
        nb.act[s][d] = act[s];
    }
    // conserved: the epoch of the owner's current buffer (the caller subtracts
    // it from the step's cumulative shift once that is known)
    for (int f = 0; f < kMaxFields; f++) nb.shift[f][d] = (cons && f == 0) ? (par[0] ? e1 : e0) : 0.0;
}

// End of a run of n >= 1 single-launch steps: the state the worklist path and
// the host read, from the per-tile bytes of the last step. Awake bitmap = the
// dilation of the last detector bits, parity bitmap, detector bytes (a tile
// that did not fire holds 0, the invariant the finalize's dilation relies on),
// steps, cell updates, the awake count, and the simulated time advanced step by
// step as the finalize advances it. One thread per tile of a segment (the
// segment starts on a 64-tile word); returns, in every thread, the segment's
// cell updates and awake-tile count.
__device__ __forceinline__ void dense_canon_seg(CInst& I, int t0, int ntile, int n, unsigned long long* scells,
                                                int* scnt, unsigned long long* cells_out, int* cnt_out) {
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int nt = I.nt, ntx = I.ntx;
    const int t = t0 + tid;
    const bool valid = tid < ntile;
    const bool regular = I.mode == 0;
    const int last = n & 1;
    const int nsets = I.nsets;
    const int nw = (ntile + 63) >> 6;
    // every load first, unconditionally (a thread past the segment reads tile t0,
    // a one-set instance reads set 0 twice; neither result is used), so they are
    // in flight together instead of waited for one branch at a time
    const int tc = valid ? t : t0;
    const int tj = tc / ntx, ti = tc - tj * ntx;
    const Nb2 nbr = nb2_of(ti, tj, ntx, I.nty, I.bc_x, I.bc_y);
    const gu8 *F, *P;
    dense_bytes(I, last, &F, &P);
    const int r0 = I.druns[tc];
    int fv[2], pv[2], av[2];
    for (int s = 0; s < 2; s++) {
        const int so = s < nsets ? s * nt : 0;
        fv[s] = F[so + tc];
        pv[s] = P[so + tc];
        av[s] = regular ? 1 : dilated2d(F + so, ti, tj, ntx, nbr);
    }
    const int r = valid ? r0 : 0;
    uint64_t wa = 0ull;
    for (int s = 0; s < nsets; s++) {
        const int f = valid ? fv[s] : 0, p = valid ? pv[s] : 0, a = valid ? av[s] : 0;
        if (valid) I.nflag[s][t] = (uint8_t)f;
        const uint64_t ws = __ballot(a), wp = __ballot(p);
        wa |= ws;
        if (lane == 0 && wid < nw) {
            I.par[s][(t0 >> 6) + wid] = wp;
            if (!regular) I.a_cur[s][(t0 >> 6) + wid] = ws;
        }
    }
    if (valid) I.druns[t] = 0;
    unsigned long long cells =
        valid ? (unsigned long long)r * (unsigned long long)(I.full_tiles ? I.tx * I.ty * I.tz : tile_cells(I, t))
              : 0ull;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) cells += __shfl_down(cells, off, 64);
    if (lane == 0) {
        scells[wid] = cells;
        scnt[wid] = __popcll(wa);
    }
    __syncthreads();
    unsigned long long c = 0;
    int cnt = 0;
    for (int w = 0; w < nw; w++) {
        c += scells[w];
        cnt += scnt[w];
    }
    *cells_out = c;
    *cnt_out = cnt;
}

// The instance counters after n single-launch steps (one thread).
__device__ __forceinline__ void dense_canon_finish(CInst& I, int n, unsigned long long cells, int64_t cnt) {
    I.ctr[0] = I.ctr[0] + n;
    I.ctr[1] = I.ctr[1] + (int64_t)cells;
    I.ctr[2] = cnt;
    const double dt = I.scal[1];
    double tm = I.scal[2];
    for (int i = 0; i < n; i++) tm += dt;
    I.scal[2] = tm;
    I.scal[3] = dt;
}

// After a resident launch (res: its state and count, k_resident.h; null after single-launch
// steps): whether it was given up. Then its steps are counted in ctr[3], for the host,
// and everything else stays as it was before them.
__device__ __forceinline__ bool resident_given_up(const uint32_t* res) { return res && res[0] == 1u; }

__device__ __forceinline__ void resident_skip_seg(CInst& I, int t0, int ntile) {
    if ((int)threadIdx.x < ntile) I.druns[t0 + threadIdx.x] = 0;
}

// One instance in one segment: one workgroup does it all. Conserved (CH): the
// cumulative shift after the last step, from the last step's change sums in the
// finalize's order (block_sum over the tiles, 0 for tiles that did not run).
__global__ __launch_bounds__(kFinNT) void dense_canon_kernel(const Inst* __restrict__ insts, int n, uint32_t* res) {
    __shared__ unsigned long long scells[kFinNT / 64];
    __shared__ int scnt[kFinNT / 64];
    __shared__ double sd[kFinNT / 64 + 1];
    CInst& I = ((CInst*)insts)[0];
    if (resident_given_up(res)) {
        resident_skip_seg(I, 0, I.nt);
        if (threadIdx.x == 0) I.ctr[3] += n;
        return;
    }
    unsigned long long c;
    int cnt;
    dense_canon_seg(I, 0, I.nt, n, scells, scnt, &c, &cnt);
    if (I.mode == 2) {
        const int last = n & 1, t = threadIdx.x;
        const double v = t < I.nt ? I.tpart[(int64_t)(1 + last) * I.nt + t] : 0.0;
        const double tot = block_sum<kFinNT>(v, sd);
        if (t == 0) I.scal[8] = I.scal[12 + last] + tot / I.ntotal;
    }
    if (threadIdx.x == 0) {
        dense_canon_finish(I, n, c, cnt);
        if (res) res[0] = res[1] = 0u;  // (every thread read it before the segment's barrier)
    }
}

// Several segments or instances: one workgroup per segment writes its partial
// sums (parts[seg].cells, counts[seg]) ...
__global__ __launch_bounds__(kFinNT) void dense_canon_seg_kernel(const Inst* __restrict__ insts,
                                                                 const Seg* __restrict__ segs,
                                                                 SegPart* __restrict__ parts,
                                                                 int32_t* __restrict__ counts, int n,
                                                                 const uint32_t* res) {
    __shared__ unsigned long long scells[kFinNT / 64];
    __shared__ int scnt[kFinNT / 64];
    const Seg sg = segs[blockIdx.x];
    CInst& I = ((CInst*)insts)[sg.inst];
    if (resident_given_up(res)) {
        resident_skip_seg(I, sg.tile0, sg.ntile);
        return;
    }
    unsigned long long c;
    int cnt;
    dense_canon_seg(I, sg.tile0, sg.ntile, n, scells, scnt, &c, &cnt);
    if (threadIdx.x == 0) {
        parts[blockIdx.x].cells = c;
        counts[blockIdx.x] = cnt;
    }
}

// ... and one wave per instance sums them in segment order.
__global__ __launch_bounds__(kFinNT) void dense_canon_merge_kernel(const Inst* __restrict__ insts,
                                                                   const InstSegs* __restrict__ isegs, int n_inst,
                                                                   const SegPart* __restrict__ parts,
                                                                   const int32_t* __restrict__ counts, int n,
                                                                   uint32_t* res) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (resident_given_up(res)) {  // (a resident launch is one instance's)
        if (threadIdx.x == 0) ((CInst*)insts)[0].ctr[3] += n;
        return;
    }
    __syncthreads();
    if (res && threadIdx.x == 0) res[0] = res[1] = 0u;
    for (int i = wid; i < n_inst; i += kFinNT / 64) {
        const InstSegs r = isegs[i];
        unsigned long long c = 0;
        int64_t cnt = 0;
        for (int q = r.first + lane; q < r.first + r.count; q += 64) {
            c += parts[q].cells;
            cnt += counts[q];
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            c += __shfl_down(c, off, 64);
            cnt += __shfl_down(cnt, off, 64);
        }
        if (lane == 0) dense_canon_finish(((CInst*)insts)[i], n, c, cnt);
    }
}

// Current value of one field: the buffer the tile parity selects, minus the
// conserved shift accumulated since the tile last ran.
__global__ void materialize_kernel(const Inst* __restrict__ insts, int slot, int field, double* __restrict__ dst) {
    CInst& I = ((CInst*)insts)[slot];
    const int64_t n = (int64_t)I.nx * I.ny * I.nz;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = current_value(I, field, i);
}

// After an upload: both buffers hold the new values, so the shift epochs of
// every tile restart at the current cumulative shift.
__global__ void reset_epochs_kernel(const Inst* __restrict__ insts, int slot) {
    CInst& I = ((CInst*)insts)[slot];
    for (int f = 0; f < I.ncons; f++) {
        const double S = I.scal[8 + f];
        for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < 2 * I.nt; i += gridDim.x * blockDim.x)
            I.s_tile[(int64_t)f * 2 * I.nt + i] = S;
    }
}

// Non-finite check over the current values of all fields.
__global__ void finite_kernel(const Inst* __restrict__ insts, int slot, int* __restrict__ bad) {
    CInst& I = ((CInst*)insts)[slot];
    const int64_t n = (int64_t)I.nx * I.ny * I.nz;
    for (int f = 0; f < I.nfields; f++) {
        const int set = I.field_set[f];
        for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
            const int x = (int)(i % I.nx);
            const int y = (int)((i / I.nx) % I.ny);
            const int z = (int)(i / ((int64_t)I.nx * I.ny));
            const int t = x / I.tx + (y / I.ty) * I.ntx + (z / I.tz) * I.ntx * I.nty;
            const double v = I.buf[bit_of(I.par[set], t)][f][i];
            if (!isfinite(v)) atomicOr(bad, 1);
        }
    }
}

}  // namespace dba
