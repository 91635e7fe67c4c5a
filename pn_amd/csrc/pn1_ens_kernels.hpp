// pn1_ens_kernels.hpp -- device code for ensembles of independent clusters.
//
// All clusters live in one state (SoA stride cap).  Cluster c occupies
// particles [coff[c], coff[c + 1]); its BH is particle coff[c], its stars
// follow.  One force evaluation of the whole ensemble is two launches, after
// one that prepares the first (as in a single context):
//
//   k_ens_prep   per-star j-records and the clusters' separable sums;
//                workgroups come from a table, each inside one cluster, and
//                a cluster's last one adds its sums (a ticket per cluster)
//   k_ens_pair*w one launch for all clusters, a workgroup of PW waves per
//                (cluster, row of 64 stars, j chunk) of the automatic plan
//   k_ens_pair*  with an explicit chunk length or kernel variant: one
//                persistent launch for all clusters: workgroups take
//                (cluster, 256-star i-block, j-chunk) items from per-XCD
//                queues (atomic counters), items sorted by decreasing cost
//                on the host; every item writes its partial sums to its own
//                slot, so the result does not depend on which workgroup ran
//                which item
//   k_ens_fin    per row of 64 stars, as k_fin, with its cluster's sums and
//                BH; it also resets the pair kernel's queues
//
// The pair arithmetic is the single-cluster kernels' (body64 / body32),
// and so is the order of each lane's j loop: with one chunk per cluster
// the results equal a single-cluster run with an unsplit j range bit for
// bit.
//
// Included by pn1_api.hip and pn1_pair32.hip (the mixed-form pair kernels):
// the kernels that are not templates are declared inline.
#pragma once
#include "pn1_ens_types.hpp"
#include "pn1_kernels.hpp"

namespace pn1dev {

// Lane geometry of an item: the lane's local star, its particle index
// (clamped into the cluster for lanes past its end) and the wave's own
// window [w0, w1) of the chunk (masked self pairs).
struct EGeom {
    int li, i, w0, w1;
    bool live;   // the wave holds at least one of the cluster's stars
};

__device__ __forceinline__ EGeom ens_geom(const EItem& w)
{
    EGeom g;
    g.li = w.ib * WG + (int)threadIdx.x;
    g.i = w.off + 1 + (g.li < w.nst ? g.li : w.nst - 1);
    const int wl = w.ib * WG + (__builtin_amdgcn_readfirstlane((int)threadIdx.x) & ~63);
    const int wb = w.off + 1 + wl;
    g.w0 = max(w.j0, wb);
    g.w1 = min(w.j1, wb + 64);
    g.live = wl < w.nst;
    return g;
}

template <int PP>
__device__ __forceinline__ void ens_pair64(const JRec64* __restrict__ jr,
                                           const double* __restrict__ st,
                                           double* __restrict__ part,
                                           const EItem* __restrict__ items,
                                           unsigned int* __restrict__ counter,
                                           const int* __restrict__ qoff, Phys P)
{
    int q = 0;
    for (;;) {
        const int it = ens_take(counter, qoff, q);
        if (it < 0) break;
        const EItem w = items[it];
        const EGeom g = ens_geom(w);
        const I64 I = load_i64(jr, st, P.cap, g.i, P.eps2);
        // a wave past the cluster's last star (a partly filled last i
        // block) skips the loop: it would only repeat that star's sums
        if (!g.live) continue;
        double a[NACC];
#pragma unroll
        for (int k = 0; k < NACC; ++k) a[k] = 0.0;
        if (g.w0 < g.w1) {
            run64<false, PP>(jr, w.j0, g.w0, g.i, I, a, P.eps2);
            run64<true, PP>(jr, g.w0, g.w1, g.i, I, a, P.eps2);
            run64<false, PP>(jr, g.w1, w.j1, g.i, I, a, P.eps2);
        } else {
            run64<false, PP>(jr, w.j0, w.j1, g.i, I, a, P.eps2);
        }
        if (g.li < w.nst) {
            double* pp = part + w.pslot * NACC + g.li;
#pragma unroll
            for (int k = 0; k < NACC; ++k) stream_out(a[k], &pp[(size_t)k * w.nst]);
        }
    }
}

template <int PP, bool TS, bool EQ>
__device__ __forceinline__ void ens_pair32(const JRec32* __restrict__ jr,
                                           const JRec64* __restrict__ j64,
                                           const Thr* __restrict__ thr,
                                           const double* __restrict__ st,
                                           float* __restrict__ part,
                                           const EItem* __restrict__ items,
                                           unsigned int* __restrict__ counter,
                                           const int* __restrict__ qoff,
                                           const double* __restrict__ cmmax, Phys P, int tile)
{
    int q = 0;
    for (;;) {
        const int it = ens_take(counter, qoff, q);
        if (it < 0) break;
        const EItem w = items[it];
        const EGeom g = ens_geom(w);
        const I32 I = load_i32(j64, thr, st, P.cap, g.i, w.off, P.eps2);
        if (!g.live) continue;                 // as in k_ens_pair64
        float a[NACC32], sN[3], cN[3];
#pragma unroll
        for (int k = 0; k < NACC32; ++k) a[k] = 0.0f;
#pragma unroll
        for (int k = 0; k < 3; ++k) sN[k] = cN[k] = 0.0f;
        int cnt = 0;
        const float e2 = P.eps2f;
        const double e2d = P.eps2, rs = 1.0 / cmmax[w.c];
        if (g.w0 < g.w1) {
            run32<false, PP, TS, EQ>(jr, j64, w.j0, g.w0, g.i, I, a, e2, e2d, rs, sN, cN, tile, cnt);
            run32<true, PP, TS, EQ>(jr, j64, g.w0, g.w1, g.i, I, a, e2, e2d, rs, sN, cN, tile, cnt);
            run32<false, PP, TS, EQ>(jr, j64, g.w1, w.j1, g.i, I, a, e2, e2d, rs, sN, cN, tile, cnt);
        } else {
            run32<false, PP, TS, EQ>(jr, j64, w.j0, w.j1, g.i, I, a, e2, e2d, rs, sN, cN, tile, cnt);
        }
        fold_newton(a, sN, cN);
        if (g.li < w.nst) {
            float* pp = part + w.pslot * MROWS + g.li;
#pragma unroll
            for (int k = 0; k < NACC32; ++k)
                if (TS || k != A_TS) stream_out(k <= A_NZ ? sN[k] : a[k], &pp[(size_t)k * w.nst]);
#pragma unroll
            for (int k = 0; k < 3; ++k) stream_out(cN[k], &pp[(size_t)(NACC32 + k) * w.nst]);
        }
    }
}

// The kernels.  The persistent loop keeps an item's geometry live beside
// the pair sums, which left to itself the compiler pays for with registers
// (66 to 99 VGPRs, 4 to 7 waves per SIMD against the single-cluster
// kernels' 60 and 72).  The forms with one j-record at a time are held to
// the single-cluster kernels' occupancy: 8 waves per SIMD for the mixed
// kernel (64 VGPRs, no spills), 7 for the FP64 one; the two-in-flight forms
// (variant bit 0) are left to the compiler, which would spill them there.
template <int PP>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(7, 8)))
void k_ens_pair64(const JRec64* __restrict__ jr, const double* __restrict__ st,
                  double* __restrict__ part, const EItem* __restrict__ items,
                  unsigned int* __restrict__ counter, const int* __restrict__ qoff, Phys P)
{
    ens_pair64<PP>(jr, st, part, items, counter, qoff, P);
}

template <int PP>
__global__ __launch_bounds__(WG)
void k_ens_pair64x(const JRec64* __restrict__ jr, const double* __restrict__ st,
                   double* __restrict__ part, const EItem* __restrict__ items,
                   unsigned int* __restrict__ counter, const int* __restrict__ qoff, Phys P)
{
    ens_pair64<PP>(jr, st, part, items, counter, qoff, P);
}

template <int PP, bool TS, bool EQ>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(8, 8)))
void k_ens_pair32(const JRec32* __restrict__ jr, const JRec64* __restrict__ j64,
                  const Thr* __restrict__ thr, const double* __restrict__ st,
                  float* __restrict__ part, const EItem* __restrict__ items,
                  unsigned int* __restrict__ counter, const int* __restrict__ qoff,
                  const double* __restrict__ cmmax, Phys P, int tile)
{
    ens_pair32<PP, TS, EQ>(jr, j64, thr, st, part, items, counter, qoff, cmmax, P, tile);
}

template <int PP, bool TS, bool EQ>
__global__ __launch_bounds__(WG)
void k_ens_pair32x(const JRec32* __restrict__ jr, const JRec64* __restrict__ j64,
                   const Thr* __restrict__ thr, const double* __restrict__ st,
                   float* __restrict__ part, const EItem* __restrict__ items,
                   unsigned int* __restrict__ counter, const int* __restrict__ qoff,
                   const double* __restrict__ cmmax, Phys P, int tile)
{
    ens_pair32<PP, TS, EQ>(jr, j64, thr, st, part, items, counter, qoff, cmmax, P, tile);
}

// ---------------------------------------------------------------------
// the automatic plan: k_pair64w and k_pair32w over a table of (cluster, row,
// chunk)
// ---------------------------------------------------------------------
// Item k of queue q is workgroup sum_q' min(k, len q') + (queues before q with
// more than k items): the queues side by side, so that workgroup b, which the
// dispatcher gives to XCD b % 8, takes an item of queue b % 8 until the
// shortest queue ends.  A queue holds whole clusters, those with the longest
// parts first.  A workgroup per cluster.
inline __global__ __launch_bounds__(WG) void k_ens_parts(const EPlace* __restrict__ place, int nc,
                                                        const int* __restrict__ crow, QLen len,
                                                        EPart* __restrict__ parts)
{
    const int c = ens_block();
    if (c >= nc) return;
    const EPlace w = place[c];
    const int cnt = (crow[c + 1] - crow[c]) * w.S;       // S = 0: no star
    for (int t = threadIdx.x; t < cnt; t += WG) {
        const int k = w.k0 + t;
        int b = 0;
#pragma unroll
        for (int q = 0; q < NXCD; ++q) b += min(k, len.n[q]) + (q < w.q && len.n[q] > k ? 1 : 0);
        parts[b] = EPart{c, t / w.S, t % w.S, w.S};
    }
}

// The item's cluster (BH at off, nst stars), its lane's star li (particle i,
// clamped) and wave's records R.
struct EWave {
    int off, nst, li, i;
    JRange R;
};

__device__ __forceinline__ EWave ens_wave(const EPart& w, const int* __restrict__ coff, int wave,
                                          int lane)
{
    EWave g;
    g.off = coff[w.c];
    g.nst = coff[w.c + 1] - g.off - 1;
    g.li = w.ig * RB + lane;
    g.i = g.off + 1 + min(g.li, g.nst - 1);
    const int len = (g.nst + w.S * PW - 1) / (w.S * PW), j0 = g.off + 1;
    g.R.j0 = j0 + min(g.nst, (w.s * PW + wave) * len);
    g.R.j1 = j0 + min(g.nst, (w.s * PW + wave + 1) * len);
    g.R.w0 = max(g.R.j0, j0 + w.ig * RB);
    g.R.w1 = min(g.R.j1, j0 + w.ig * RB + RB);
    return g;
}

inline __global__ __launch_bounds__(PW * RB) __attribute__((amdgpu_waves_per_eu(7, 8)))
void k_ens_pair64w(const JRec64* __restrict__ jr, const double* __restrict__ st,
                   double* __restrict__ part, const EPart* __restrict__ parts,
                   const int* __restrict__ coff, const long long* __restrict__ poff, Phys P)
{
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const EPart w = parts[blockIdx.x];
    const EWave g = ens_wave(w, coff, wave, lane);
    const I64 I = load_i64(jr, st, P.cap, g.i, P.eps2);
    double a[NACC];
    part64(jr, g.R, g.i, I, a, P.eps2);
    double t[NSHARE<NACC>];
    waves_share(a, wave, lane, t);
    if (g.li < g.nst) {
        double* pp = part + (poff[w.c] + (long long)w.s * g.nst) * NACC + g.li;
#pragma unroll
        for (int q = 0; q < NSHARE<NACC>; ++q)
            stream_out(t[q], &pp[(size_t)(q * PW + wave) * g.nst]);
    }
}

template <bool TS, bool EQ>
__global__ __launch_bounds__(PW * RB) __attribute__((amdgpu_waves_per_eu(8, 8)))
void k_ens_pair32w(const JRec32* __restrict__ jr, const JRec64* __restrict__ j64,
                   const Thr* __restrict__ thr, const double* __restrict__ st,
                   float* __restrict__ part, const EPart* __restrict__ parts,
                   const int* __restrict__ coff, const long long* __restrict__ poff,
                   const double* __restrict__ cmmax, Phys P, int tile,
                   const int* __restrict__ crow, const unsigned long long* __restrict__ hmask,
                   double* __restrict__ hpart)
{
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const EPart w = parts[blockIdx.x];
    const EWave g = ens_wave(w, coff, wave, lane);
    const I32 I = load_i32(j64, thr, st, P.cap, g.i, g.off, P.eps2);
    float a[NACC32], sumN[3], cmpN[3];
    part32<TS, EQ>(jr, j64, g.R, g.i, I, P.eps2f, P.eps2, 1.0 / cmmax[w.c], tile, a, sumN, cmpN);
    put_part32<TS>(a, sumN, cmpN, wave, lane, g.li < g.nst,
                   part + (poff[w.c] + (long long)w.s * g.nst) * MROWS + g.li, (size_t)g.nst);
    if (hpart && w.S <= HCHUNK) {
        const int row = crow[w.c] + w.ig;
        const unsigned long long hm = hmask[row];
        if (hm) {
            const EWave a = ens_wave(w, coff, 0, lane), b = ens_wave(w, coff, PW - 1, lane);
            hard_part(j64, st, P.cap, P.eps2, g.off + 1 + w.ig * RB, hm, a.R.j0, b.R.j1,
                      hpart + ((size_t)row * HSLOT * HCHUNK + w.s) * (NACC + 1));
        }
    }
}

// Per-cluster buffers.  Cluster c's rows of 64 stars are [crow[c],
// crow[c + 1]) (at least one, also without stars).
struct EnsBufs {
    const double* cm0;
    const int* coff;
    const int* crow;
    const double *cmmax, *ctauf;
    unsigned int* counter;        // the pair kernel's queues
};

__device__ __forceinline__ void reset_queues(unsigned int* counter)
{
    if (ens_block() == 0 && threadIdx.x < NXCD) counter[threadIdx.x] = 0u;
}

// As k_prep, one workgroup per FG rows of a cluster (pblk: its cluster and
// first local star).  M.mmax, M.tauf: per cluster, from E; R.ticket, R.gs and
// R.fn: one entry (or NGS) per cluster.
inline __global__ __launch_bounds__(FWG) void k_ens_prep(const double* __restrict__ st,
                                                const double* __restrict__ m, Phys P, EnsBufs E,
                                                const EBlk* __restrict__ pblk, int npblk,
                                                JRec64* __restrict__ j64, RowBufs R, MixPrep M,
                                                const double* __restrict__ aprev,
                                                const float* __restrict__ kprev)
{
    reset_queues(E.counter);
    const int wg = ens_block();
    if (wg >= npblk) return;
    const EBlk b = pblk[wg];
    const int off = E.coff[b.c], nst = E.coff[b.c + 1] - off - 1;
    const int r0 = E.crow[b.c], r1 = E.crow[b.c + 1];
    const int row = r0 + b.first / RB + (int)(threadIdx.x >> 6);
    const size_t cap = (size_t)P.cap;
    if (M.j32) {
        M.mmax = E.cmmax[b.c];
        M.tauf = E.ctauf[b.c];
    }
    if (row < r1) {
        const int li = b.first + (int)threadIdx.x;
        double g[NGS];
        bool f = false, hard = false;
        const bool ok = li < nst;
        if (ok) {
            const int p = off + 1 + li;
            const double x[3] = {st[p], st[cap + p], st[2 * cap + p]};
            const double v[3] = {st[3 * cap + p], st[4 * cap + p], st[5 * cap + p]};
            const double x0[3] = {st[off], st[cap + off], st[2 * cap + off]};
            double a[3] = {0.0, 0.0, 0.0};
            float kr = 0.0f;
            if (aprev) {
#pragma unroll
                for (int k = 0; k < 3; ++k) a[k] = aprev[k * cap + p];
                kr = kprev[p];
            }
            f = prep_star(x, v, x0, m[p], p, E.cm0[b.c], P.eps2, j64, g, M, aprev != nullptr, a,
                          kr, hard);
        }
        const double cb[3] = {0.0, 0.0, 0.0};
        put_row<false, true>(row, 0, ok, cb, g, R.rows, M.j32 != nullptr, f, hard, R.fmask,
                             R.hnext);
    }
    if (last_block(R.ticket + b.c, (unsigned)((r1 - r0 + FG - 1) / FG)))
        close_prep(R, M.j32 != nullptr, r0, r1, off + 1, R.gs + (size_t)b.c * NGS, R.flist + off,
                   R.fn + b.c);
}

// As k_fin: one workgroup per row of the ensemble (G = FG, blk the row
// table) or per FG rows of a cluster (G = 1, blk = pblk), n in all.
template <int MODE, int STAGE, int G>
__global__ __launch_bounds__(FWG) __attribute__((amdgpu_waves_per_eu(4, 8)))
void k_ens_fin(FinBufs F, RowBufs R, EnsBufs E, const EBlk* __restrict__ blk, int n,
               const void* __restrict__ part, const long long* __restrict__ poff, int L,
               MixPrep M, Phys P)
{
    reset_queues(E.counter);
    const int wg = ens_block();
    if (wg >= n) return;
    const EBlk b = blk[wg];
    const int off = E.coff[b.c], nst = E.coff[b.c + 1] - off - 1;
    const int r0 = E.crow[b.c], r1 = E.crow[b.c + 1];
    const Row q = {off, nst, b.first, r0 + b.first / RB, nst};
    double* gs = R.gs + (size_t)b.c * NGS;
    if (MODE == 1) {
        M.mmax = E.cmmax[b.c];
        M.tauf = E.ctauf[b.c];
    }
    StageIn bh = {};
    if (nst > 0) {
        if (ens_nchunks(nst, L) > HCHUNK) F.hp = nullptr;
        const void* base = MODE == 0 ? (const void*)((const double*)part + poff[b.c] * NACC)
                                     : (const void*)((const float*)part + poff[b.c] * MROWS);
        fin_rows<MODE, STAGE, G, 1>(F, R, q, base, ens_nchunks(nst, L), (size_t)nst, 0, gs,
                                 R.flist + off, R.fn + b.c, E.cm0[b.c], M, P, bh, 0);
    } else {
        empty_row<1>(R, q.row, MODE == 1);
    }
    const unsigned nblk = (unsigned)(G == 1 ? (r1 - r0 + FG - 1) / FG : r1 - r0);
    if (last_block(R.ticket + b.c, nblk)) {
        if (G > 1 && nst > 0)
            fin_close<MODE, STAGE, true, 1>(F, R, r0, r1, off, gs, R.flist + off, R.fn + b.c, P, bh);
        else
            fin_close<MODE, STAGE, false, 1>(F, R, r0, r1, off, gs, R.flist + off, R.fn + b.c, P, bh);
    }
}

// ---------------------------------------------------------------------
// ensemble energies (FP64)
// ---------------------------------------------------------------------
// As k_energy, workgroup (row of the ensemble, chunk); a cluster uses
// energy_chunks of the grid's chunks, the others leave at once (the grid's third
// dimension: further rows).  Its last workgroup writes its energies to out[5 c].
inline __global__ __launch_bounds__(PW * RB)
void k_ens_energy(const JRec64* __restrict__ jr, const double* __restrict__ st, EnsBufs E,
                  const EBlk* __restrict__ rowt, int nrows, const double* __restrict__ gs,
                  double* __restrict__ eb, double* __restrict__ out,
                  unsigned int* __restrict__ ticket, Phys P)
{
    __shared__ double t[EV];
    const int2 w = energy_item();
    const int r = (int)(blockIdx.z * gridDim.x) + w.x, s = w.y;
    if (r >= nrows) return;
    const int c = rowt[r].c;
    const int off = E.coff[c], nst = E.coff[c + 1] - off - 1;
    const int S = energy_chunks(nst), r0 = E.crow[c], nrow = E.crow[c + 1] - r0;
    if (s >= S) return;
    const double m0 = E.cm0[c], G1 = gs[(size_t)c * NGS + G_G1];
    if (nst > 0)
        energy_row(jr, st, P.cap, off, nst, nrow, r - r0, s, S, m0, G1, P.eps2, t);
    else if (threadIdx.x < EV)
        t[threadIdx.x] = 0.0;
    if (threadIdx.x < EV)
        hand_over(&eb[((size_t)r * ECHUNK + s) * EV + threadIdx.x], t[threadIdx.x]);
    if (last_block(ticket + c, (unsigned)(nrow * S)))
        energy_total(eb + (size_t)r0 * ECHUNK * EV, nrow * S, S, ECHUNK, st, P.cap, off, m0, G1,
                     P.lam, out + (size_t)c * 5);
}

}  // namespace pn1dev
