// pn1_kernels.hpp -- device code of libpn1 (gfx950, wave64).
//
// One force evaluation of Limit-sticky9's force() (Limit-sticky9.c:21-424)
// is two launches on one stream, after one that prepares the first:
//
//   k_prep    O(n)   per-star BH geometry (d, |d|^2, e = (|d|^2+eps^2)^-1/2)
//                    written once as an AoS j-record, and the separable sums
//                    (sum m e, sum m e^3 d, ...)
//   k_pair*   O(n^2) the star-star pair sums, one rsqrt per pair
//   k_fin     O(n)   star accelerations from the pair sums and the O(n)
//                    closed forms, the BH's acceleration, the stage update of
//                    the RK driver and, inside a step, all that k_prep does
//                    for the driver's next evaluation
//
// A step of the driver is therefore k_prep once and then (k_pair, k_fin)
// three times per step.  The O(n) kernels end with the sums over all stars:
// their workgroups take a ticket when done, and the last one adds the
// per-row partials and finishes the BH (last_block).
//
// Pair kernels: i-particle per lane in VGPRs; the j loop has wave-uniform
// bounds, so each j-record is fetched with scalar loads into SGPRs and
// broadcast to all 64 lanes as an instruction operand (no LDS traffic in
// the inner loop).  The j range is split into S chunks (one partial per
// chunk, reduced in fixed order by k_fin), and workgroups are mapped so that
// each XCD works on one chunk, whose records then stay in that XCD's L2.
//
// All reductions use a fixed order, so results are bitwise reproducible
// for a given launch shape.
//
// Two translation units include this header: pn1_api.hip launches every
// kernel but the mixed-form pair kernels, pn1_pair32.hip those.  The kernels
// that are not templates are therefore declared inline.
#pragma once
#include "pn1_common.hpp"
#include "pn1_rows.hpp"

namespace pn1dev {
// What the stage update of the reference's RK driver (Limit-sticky9.c:853-891)
// reads of particle p: its state in this force call (x, v) and, from stage 2
// on, at the start of the step (X, V); stage 3 also the sums of the two
// stage states (hx, hv).  Loaded ahead of the acceleration it needs.
struct StageIn {
    double x[3], v[3], X[3], V[3], hx[3], hv[3];
};

// Of components row0 .. row0 + n - 1, in s from index 0 on.
template <int STAGE>
__device__ __forceinline__ StageIn stage_load(const double* in, const double* X,
                                              const double* H1, const double* H2, int cap, int p,
                                              int row0 = 0, int n = 3)
{
    StageIn s;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        if (k >= n) break;
        const size_t ix = (size_t)(row0 + k) * cap + p, iv = (size_t)(3 + row0 + k) * cap + p;
        s.x[k] = in[ix];
        s.v[k] = in[iv];
        if (STAGE >= 2) {
            s.X[k] = X[ix];
            s.V[k] = X[iv];
        }
        if (STAGE == 3) {
            s.hx[k] = H1[ix] + H2[ix];
            s.hv[k] = H1[iv] + H2[iv];
        }
    }
    return s;
}

// The position the driver's next force call takes (its velocities are known
// before this call's acceleration), component k.  FMA contraction is off
// here and below so each line rounds exactly as the reference's.
template <int STAGE>
__device__ __forceinline__ double stage_pos(const StageIn& s, double dt, int k)
{
#pragma clang fp contract(off)
    if (STAGE == 1) return s.x[k] + 0.5 * s.v[k] * dt;
    if (STAGE == 2) return s.X[k] + 0.5 * s.v[k] * dt;   // v1 of stage 1
    if (STAGE == 3) {
        const double hx3 = s.X[k] + s.v[k] * dt;         // v1 of stage 2
        return (s.X[k] + hx3 + 2.0 * s.hx[k]) / 6.0;
    }
    return s.x[k];
}

// Stage update of component k of particle p (row `row` of the SoA state, k
// of s), given its acceleration a; STAGE 1..3 follow the three force calls,
// STAGE 0 (plain force evaluation) does nothing.  nx, nv receive the state
// the driver's next force call takes (Y after stages 1 and 2, X after
// stage 3).
template <int STAGE>
__device__ __forceinline__ void stage_update(int p, int cap, const StageIn& s, int k, int row,
                                             double a, double* X, double* Y, double* H1,
                                             double* H2, double dt, double& nx, double& nv)
{
#pragma clang fp contract(off)
    if (STAGE == 0) return;
    const size_t ix = (size_t)row * cap + p, iv = (size_t)(3 + row) * cap + p;
    nx = stage_pos<STAGE>(s, dt, k);
    if (STAGE == 1) {
        nv = s.v[k] + 0.5 * a * dt;
        Y[ix] = nx; Y[iv] = nv; H1[ix] = nx; H1[iv] = nv;
    } else if (STAGE == 2) {
        nv = s.V[k] + 0.5 * a * dt;
        Y[ix] = nx; Y[iv] = nv; H2[ix] = nx; H2[iv] = nv;
    } else {
        const double hv3 = s.V[k] + a * dt;
        nv = (s.V[k] + hv3 + 2.0 * s.hv[k]) / 6.0;
        X[ix] = nx;
        X[iv] = nv;
    }
}

// ---------------------------------------------------------------------
// k_prep: per-star BH geometry + separable sums
// ---------------------------------------------------------------------
// Mixed form's pair thresholds of a star at x from its BH whose previous
// evaluation gave the acceleration a and cancellation ratio kr (known:
// false if there was none), for star masses up to mmax (see Thr).
__device__ __forceinline__ Thr pair_thresholds(const double (&x)[3], bool known,
                                               const double (&a)[3], float kr, double mmax,
                                               bool& hard)
{
    Thr t;
    hard = false;
    if (!known) {
        t.rc2 = 0.0f;
        t.dn2 = __FLT_MAX__;
        return t;
    }
    hard = !(kr <= (float)PN1_HARD_K);                         // NaN too
    if (hard) {                  // the FP32 lane's sums are not used
        t.rc2 = t.dn2 = 0.0f;
        return t;
    }
    // 1 / |a| and |x| from one reciprocal square root each, and the power
    // 2/3 from the FP32 logarithm and exponential (dn2 to ~1e-6: it only says
    // where the lo parts start to matter)
    const double A2 = a[0] * a[0] + a[1] * a[1] + a[2] * a[2];
    const double X2 = x[0] * x[0] + x[1] * x[1] + x[2] * x[2];
    const double q = mmax * rsq64(A2);                          // NaN if A2 == 0
    const float rc2 = (float)fmin(q * (1.0 / PN1_CLOSE_KAPPA), (double)__FLT_MAX__);
    const float dn3 = (float)(6.0 * 0x1p-24 / PN1_LAZY_ETA * q * (X2 * rsq64(X2)));
    const float dn2 = __builtin_amdgcn_exp2f((2.0f / 3.0f) * __builtin_amdgcn_logf(dn3));
    t.rc2 = rc2;
    // no acceleration to compare with: every pair is close
    t.dn2 = A2 > 0.0 ? fmaxf(fminf(dn2, __FLT_MAX__), rc2) : __FLT_MAX__;
    return t;
}

// Star p at x, velocity v, of a cluster whose BH sits at x0 and has mass m0:
// writes its j-records and its terms of the separable sums, g.  Mixed form
// (M.j32 set): also its pair thresholds, from its previous acceleration a
// and cancellation ratio kr (`known`: there was one), and its mixed record
// in units of the cluster's largest star mass M.mmax; returns whether the
// star is close enough to the BH to be taken out of the FP32 pass (see
// PN1_FLAG_ETA), in which case its mixed record is neutral; hard: whether
// its pair terms cancel beyond PN1_HARD_K.
__device__ __forceinline__ bool prep_star(const double (&xp)[3], const double (&vp)[3],
                                          const double (&x0)[3], double mp, int p, double m0,
                                          double eps2, JRec64* __restrict__ j64,
                                          double (&g)[NGS], const MixPrep& M, bool known,
                                          const double (&a)[3], float kr, bool& hard)
{
#pragma clang fp contract(off)
    hard = false;
    const double x = xp[0], y = xp[1], z = xp[2], vx = vp[0], vy = vp[1], vz = vp[2];
    const double dx = x - x0[0], dy = y - x0[1], dz = z - x0[2];
    const double D2 = dx * dx + dy * dy + dz * dz;
    const double e = rsq64(D2 + eps2);
    const double E3 = e * e * e;
    const double q = mp * E3;
    const double V2 = vx * vx + vy * vy + vz * vz;
    JRec64 r;
    r.x = x; r.y = y; r.z = z;
    r.sx = PN1_SQ15 * vx; r.sy = PN1_SQ15 * vy; r.sz = PN1_SQ15 * vz;
    r.m = mp; r.D2 = D2;
    r.A = 1.25 * m0 * e - 2.0 * V2; r.B = 0.25 * m0 * E3;
    const double Q = 3.5 * m0 * q;
    r.MB = mp * r.B;
    r.Qdx = Q * dx; r.Qdy = Q * dy; r.Qdz = Q * dz;
    r.e = e; r.Ae = 1.5 * V2 + m0 * e;
    j64[p] = r;
    g[G_G1] = mp * e;
    g[G_M1X] = q * dx; g[G_M1Y] = q * dy; g[G_M1Z] = q * dz;
    g[G_PX] = mp * vx; g[G_PY] = mp * vy; g[G_PZ] = mp * vz;
    if (!M.j32) return false;
    const bool flagged = M.lam * mp * e * e > M.tauf;
    JRec32 h;
    if (flagged) {
        // far away (w ~ 1e-18: every FP32 pair term vanishes), no mass and
        // no 1PN fields (t = |r|^2 - D2_i is then ~1e36)
        h.xh = h.yh = h.zh = PN1_FAR;
        h.xl = h.yl = h.zl = 0.0f;
        h.sx = h.sy = h.sz = 0.0f;
        h.m = 0.0f;
        h.A = h.B = h.MB = 0.0f;
        h.Qdx = h.Qdy = h.Qdz = 0.0f;
    } else {
        // double-single position relative to the BH: the FP32 hi parts then
        // round at the cluster's own scale, wherever the cluster sits
        h.xh = (float)dx; h.yh = (float)dy; h.zh = (float)dz;
        h.xl = (float)(dx - (double)h.xh);
        h.yl = (float)(dy - (double)h.yh);
        h.zl = (float)(dz - (double)h.zh);
        h.sx = (float)r.sx; h.sy = (float)r.sy; h.sz = (float)r.sz;
        h.m = M.mmax > 0.0 ? (float)(mp / M.mmax) : 0.0f;     // no scale: massless stars
        h.A = (float)r.A; h.B = (float)r.B; h.MB = (float)r.MB;
        h.Qdx = (float)r.Qdx; h.Qdy = (float)r.Qdy; h.Qdz = (float)r.Qdz;
    }
    M.j32[p] = h;
    const double d[3] = {dx, dy, dz};
    M.thr[p] = pair_thresholds(d, known, a, kr, M.mmax, hard);
    return flagged;
}

// One row of stars' share of the sums over all stars, by its wave (ok: the
// lane holds a star): the BH shares cb (BH) and the separable sums g (NEXT),
// and, in the mixed form, the bit masks of its BH-close and its hard stars.
// Q = 4: the share of each of its groups of 16 stars apart; `sub` >= 0: of that
// group only, which lanes 0 .. 15 hold.
template <bool BH, bool NEXT, int Q = 1>
__device__ __forceinline__ void put_row(int row, int sub, bool ok, const double (&cb)[3],
                                        const double (&g)[NGS], double* __restrict__ rows,
                                        bool mixed, bool flagged, bool hard,
                                        unsigned long long* __restrict__ fmask,
                                        unsigned long long* __restrict__ hnext)
{
    const int lane = threadIdx.x & 63;
    double v[RV];
#pragma unroll
    for (int k = 0; k < RV; ++k) v[k] = 0.0;
    if (ok) {
        if (BH)
#pragma unroll
            for (int k = 0; k < 3; ++k) v[k] = cb[k];
        if (NEXT)
#pragma unroll
            for (int k = 0; k < NGS; ++k) v[RV_G + k] = g[k];
    }
    if (Q == 1) {
        const double t = wave_sums16(v);
        if ((lane & 3) == 0) hand_over(&rows[(size_t)row * RV + (lane >> 2)], t);
    } else {
        const double t = group_sums16(v);
        const int grp = sub < 0 ? lane / RV : sub;
        if (sub < 0 || lane < RV)
            hand_over(&rows[((size_t)row * Q + grp) * RV + (lane & (RV - 1))], t);
    }
    if (NEXT && mixed) {
        const unsigned long long f = __builtin_amdgcn_ballot_w64(ok && flagged);
        const unsigned long long h = __builtin_amdgcn_ballot_w64(ok && hard);
        if (lane == 0) {
            if (Q == 1 || sub < 0) {
                hand_over(&fmask[row], f);
                hnext[row] = h;
            } else {
                hand_over((unsigned short*)&fmask[row] + sub, (unsigned short)f);
                ((unsigned short*)&hnext[row])[sub] = (unsigned short)h;
            }
        }
    }
}

// Exclusive prefix sum of one value per thread over the workgroup (FWG
// threads), in thread order; *total receives the sum.
__device__ __forceinline__ int block_excl_scan(int v, int* total)
{
    __shared__ int wsum[FG];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    int incl = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int t = __shfl_up(incl, off, 64);
        if (lane >= off) incl += t;
    }
    if (lane == 63) wsum[wid] = incl;
    __syncthreads();
    int base = 0, all = 0;
#pragma unroll
    for (int w = 0; w < FG; ++w) {
        base += w < wid ? wsum[w] : 0;
        all += wsum[w];
    }
    *total = all;
    __syncthreads();
    return base + incl - v;
}

// The stars whose bit is set in the masks of rows [b0, b1) (row b0 starts at
// star p0), in increasing order, at out[0 ..), their number in *nout.  One
// workgroup of FWG threads.
__device__ __forceinline__ void list_flagged(const unsigned long long* mask, int b0, int b1,
                                             int p0, int* __restrict__ out,
                                             int* __restrict__ nout)
{
    int base = 0;
    for (int bb = b0; bb < b1; bb += FWG) {
        const int b = bb + (int)threadIdx.x;
        unsigned long long f = b < b1 ? take_over(&mask[b]) : 0ull;
        if (!__syncthreads_or(f != 0ull)) continue;     // hardly ever any
        int total;
        int at = base + block_excl_scan(__popcll(f), &total);
        while (f) {
            out[at++] = p0 + (b - b0) * RB + __builtin_ctzll(f);
            f &= f - 1;
        }
        base += total;
    }
    if (threadIdx.x == 0) *nout = base;
}

// The buffers of the O(n) kernels' sums over all stars.
struct RowBufs {
    double* rows;                          // per row: its RV values
    unsigned long long* fmask;             // per row: the BH-close stars of the state prepared
    const unsigned long long* hmask;       // per row: the hard stars of this evaluation
    unsigned long long* hnext;             // those of the state prepared: another buffer, because
                                           // other waves and workgroups may still read hmask
    double* gs;                            // separable sums of the evaluation
    int *flist, *fn;                       // its BH-close stars and their number
    unsigned int* ticket;                  // last_block's counter (k_prep: null if the
                                           // sums are left to k_fin_na; k_fin: null for
                                           // an i shard)
    unsigned int* clear;                   // a counter that k_prep sets to 0, or null
};

// After the last row of a prep: the separable sums, and the BH-close list of
// rows [b0, b1) (p0: row b0's first star).
template <int Q = 1>
__device__ __forceinline__ void close_prep(const RowBufs& R, bool mixed, int b0, int b1, int p0,
                                           double* __restrict__ gs, int* __restrict__ flist,
                                           int* __restrict__ fn)
{
    __shared__ double tot[RV];
    rows_total<Q>(R.rows, b0, b1, tot);
    if (threadIdx.x < NGS) gs[threadIdx.x] = tot[RV_G + threadIdx.x];
    if (mixed) list_flagged(R.fmask, b0, b1, p0, flist, fn);
}

// Records, separable sums and (mixed form) thresholds, BH-close and hard
// stars of the state st.  aprev, kprev (mixed form): each star's previous
// acceleration (SoA [3][cap]) and cancellation ratio, null after an upload.
// The BH mass is m[0].  Q: the groups whose sums k_fin adds up (one order in
// both, so that a step call continues another bit for bit).
template <int Q>
__global__ __launch_bounds__(FWG) void k_prep(const double* __restrict__ st,
                                             const double* __restrict__ m, Phys P, int nrow,
                                             JRec64* __restrict__ j64, RowBufs R, MixPrep M,
                                             const double* __restrict__ aprev,
                                             const float* __restrict__ kprev)
{
    if (R.clear && blockIdx.x == 0 && threadIdx.x == 0) *R.clear = 0u;
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * FG + (int)(threadIdx.x >> 6);
    const int p = 1 + row * RB + lane;
    const size_t cap = (size_t)P.cap;
    if (row < nrow) {
        double g[NGS];
        bool f = false, hard = false;
        const bool ok = p < P.n;
        if (ok) {
            const double x[3] = {st[p], st[cap + p], st[2 * cap + p]};
            const double v[3] = {st[3 * cap + p], st[4 * cap + p], st[5 * cap + p]};
            const double x0[3] = {st[0], st[cap], st[2 * cap]};
            double a[3] = {0.0, 0.0, 0.0};
            float kr = 0.0f;
            if (aprev) {
#pragma unroll
                for (int k = 0; k < 3; ++k) a[k] = aprev[k * cap + p];
                kr = kprev[p];
            }
            f = prep_star(x, v, x0, m[p], p, m[0], P.eps2, j64, g, M, aprev != nullptr, a, kr,
                          hard);
        }
        const double cb[3] = {0.0, 0.0, 0.0};
        put_row<false, true, Q>(row, -1, ok, cb, g, R.rows, M.j32 != nullptr, f, hard, R.fmask,
                             R.hnext);
    }
    if (R.ticket && last_block(R.ticket, gridDim.x))
        close_prep<Q>(R, M.j32 != nullptr, 0, nrow, 1, R.gs, R.flist, R.fn);
}

// ---------------------------------------------------------------------
// force pair kernel, FP64
// ---------------------------------------------------------------------
// Per-lane state of the i particle: position, g = 4 v, h = 4 v / sqrt(3/2),
// |d|^2 and |d|^2 + eps^2.
struct I64 {
    double x, y, z, gx, gy, gz, hx, hy, hz, D2e;
};

__device__ __forceinline__ I64 load_i64(const JRec64* __restrict__ jr,
                                        const double* __restrict__ st, int cap, int i,
                                        double eps2)
{
    const JRec64& r = jr[i];
    const double vx = st[3 * cap + i], vy = st[4 * cap + i], vz = st[5 * cap + i];
    I64 I;
    I.x = r.x; I.y = r.y; I.z = r.z;
    I.gx = 4.0 * vx; I.gy = 4.0 * vy; I.gz = 4.0 * vz;
    I.hx = PN1_4OSQ15 * vx; I.hy = PN1_4OSQ15 * vy; I.hz = PN1_4OSQ15 * vz;
    I.D2e = r.D2 + eps2;
    return I;
}

template <bool MASK>
__device__ __forceinline__ void body64(const JRec64& J, int j, int i, const I64& I,
                                       double (&a)[NACC], double eps2)
{
    double mj = J.m, MBj = J.MB, Qdx = J.Qdx, Qdy = J.Qdy, Qdz = J.Qdz;
    if (MASK) {
        const bool self = (j == i);
        mj = self ? 0.0 : mj;
        MBj = self ? 0.0 : MBj;
        Qdx = self ? 0.0 : Qdx;
        Qdy = self ? 0.0 : Qdy;
        Qdz = self ? 0.0 : Qdz;
    }
    const double rx = J.x - I.x, ry = J.y - I.y, rz = J.z - I.z;
    const double R2e = __builtin_fma(rx, rx, __builtin_fma(ry, ry, __builtin_fma(rz, rz, eps2)));
    const double w = rsq64(R2e);
    const double w2 = w * w;
    const double mw = mj * w;
    const double mw3 = mw * w2;
    a[A_NX] = __builtin_fma(mw3, rx, a[A_NX]);
    a[A_NY] = __builtin_fma(mw3, ry, a[A_NY]);
    a[A_NZ] = __builtin_fma(mw3, rz, a[A_NZ]);
    a[A_PHI] += mw;
    a[A_W3] += mw3;
    a[A_TX] = __builtin_fma(w, Qdx, a[A_TX]);
    a[A_TY] = __builtin_fma(w, Qdy, a[A_TY]);
    a[A_TZ] = __builtin_fma(w, Qdz, a[A_TZ]);
    const double t = R2e - I.D2e;
    a[A_ZE] = __builtin_fma(MBj, t, a[A_ZE]);
    const double sr = __builtin_fma(J.sx, rx, __builtin_fma(J.sy, ry, J.sz * rz));
    // one record operand per instruction (one scalar register pair per VALU op)
    const double tv = sr * w;
    double br = __builtin_fma(tv, tv, J.A);
    br = __builtin_fma(J.B, t, br);
    br = __builtin_fma(I.hx, J.sx, __builtin_fma(I.hy, J.sy, __builtin_fma(I.hz, J.sz, br)));
    const double Kr = mw3 * br;
    a[A_RX] = __builtin_fma(Kr, rx, a[A_RX]);
    a[A_RY] = __builtin_fma(Kr, ry, a[A_RY]);
    a[A_RZ] = __builtin_fma(Kr, rz, a[A_RZ]);
    const double gr = __builtin_fma(I.gx, rx, __builtin_fma(I.gy, ry, I.gz * rz));
    const double Ku = mw3 * __builtin_fma(-PN1_SQ6, sr, gr);
    a[A_UX] = __builtin_fma(Ku, J.sx, a[A_UX]);
    a[A_UY] = __builtin_fma(Ku, J.sy, a[A_UY]);
    a[A_UZ] = __builtin_fma(Ku, J.sz, a[A_UZ]);
    a[A_KS] += Ku;
}

// j loop.  PP bit 0 clear: one record at a time; set: two records in
// flight, the scalar loads of one issued before the other is used (j + 1 <
// j1 <= n, so jr[j + 2] stays within the cap + 2 records allocated).
// PP bit 1 (mixed form only): one Newton step on the FP32 rsqrt.
template <bool MASK, int PP>
__device__ __forceinline__ void run64(const JRec64* __restrict__ jr, int j0, int j1, int i,
                                      const I64& I, double (&a)[NACC], double eps2)
{
    if ((PP & 1) == 0) {
        for (int j = j0; j < j1; ++j) body64<MASK>(jr[j], j, i, I, a, eps2);
        return;
    }
    if (j0 >= j1) return;
    JRec64 ra = jr[j0];
    int j = j0;
    for (; j + 1 < j1; j += 2) {
        const JRec64 rb = jr[j + 1];
        body64<MASK>(ra, j, i, I, a, eps2);
        ra = jr[j + 2];
        body64<MASK>(rb, j + 1, i, I, a, eps2);
    }
    if (j < j1) body64<MASK>(ra, j, i, I, a, eps2);
}

// i blocks ib0 .. ib0 + nIblk - 1 (ib0 = 0: every star; a later first block
// evaluates one i shard of the stars against all of them).
template <int PP>
__global__ __launch_bounds__(WG) void k_pair64(const JRec64* __restrict__ jr,
                                              const double* __restrict__ st,
                                              double* __restrict__ part, Phys P, int S,
                                              int nIblk, int ib0)
{
    int s, ib;
    map_block(blockIdx.x, S, nIblk, s, ib);
    if (ib >= nIblk) return;
    ib += ib0;
    const int n = P.n;
    const int li = ib * WG + threadIdx.x + 1;
    const int i = li < n ? li : n - 1;
    const I64 I = load_i64(jr, st, P.cap, i, P.eps2);
    const JRange R = j_range(s, S, n, ib);
    const double eps2 = P.eps2;
    double a[NACC];
#pragma unroll
    for (int k = 0; k < NACC; ++k) a[k] = 0.0;
    if (R.w0 < R.w1) {
        run64<false, PP>(jr, R.j0, R.w0, i, I, a, eps2);
        run64<true, PP>(jr, R.w0, R.w1, i, I, a, eps2);
        run64<false, PP>(jr, R.w1, R.j1, i, I, a, eps2);
    } else {
        run64<false, PP>(jr, R.j0, R.j1, i, I, a, eps2);
    }
    if (li < n) {
#pragma unroll
        for (int k = 0; k < NACC; ++k) stream_out(a[k], &part[(size_t)(s * NACC + k) * P.cap + li]);
    }
}

// The automatic plan's form: a workgroup takes 64 stars, one per lane in each
// of its PW waves, and chunk s of S; wave w takes part w of the chunk (part
// s PW + w of the j range split in S PW), and the waves' sums are added
// pairwise in LDS and written as one partial.  Against one part per 256-star
// workgroup (k_pair64 / k_pair32, explicit splits) it gives short parts
// without as many partials: 16 or 24 per star instead of 64 to 128, which
// k_fin then reads in a fraction of the time, and enough waves at small n.
// Measured on MI355X, FP64 / mixed evaluation (pair and k_fin), us:
//   n         65    257   1025  2049  4097  8193     10241    32769
//   256 stars 23/31 25/29 28/31 43/60 55/56 147/98   209/130  1683/903
//   this form 12/16 13/17 16/20 24/24 44/35 120/78   181/112  1612/852
// PW = 4 and 16 were within 3% up to n = 2049; above, 16 waves leave a
// compute unit idle between workgroups (up to +30%).
constexpr int PW = 8;

// Workgroup -> chunk s of S and row ig of 64 stars, and the bounds of wave
// w's part of the chunk with the window that can contain j == i.  A split of
// TLONG + TSHORT chunks is tapered: the last TSHORT are an eighth as long and
// run after all others, so that the launch does not wait long on its last
// workgroups.  (A launch of some rows only starts at workgroup bid0 = S times
// the first row; it is never tapered.)
constexpr int TLONG = 16, TSHORT = 8;
__device__ __forceinline__ JRange j_part(int bid, int S, int nrow, int wave, int n, int& s,
                                         int& ig)
{
    const int nst = n - 1;
    int len;
    JRange R;
    if (S <= TLONG) {
        s = bid % S;
        ig = bid / S;
        len = (nst + S * PW - 1) / (S * PW);
        R.j0 = 1 + (s * PW + wave) * len;
    } else {
        const int lp = (nst + (TLONG + 1) * PW - 1) / ((TLONG + 1) * PW);
        const int t = bid - TLONG * nrow;
        if (t < 0) {
            s = bid % TLONG;
            ig = bid / TLONG;
            len = lp;
            R.j0 = 1 + (s * PW + wave) * len;
        } else {
            const int q = t % TSHORT;
            s = TLONG + q;
            ig = t / TSHORT;
            len = (lp + 7) / 8;
            R.j0 = 1 + TLONG * PW * lp + (q * PW + wave) * len;
        }
    }
    R.j0 = min(n, R.j0);
    R.j1 = min(n, R.j0 + len);
    R.w0 = max(R.j0, ig * RB + 1);
    R.w1 = min(R.j1, ig * RB + 1 + RB);
    return R;
}

// Adds the waves' v pairwise in a fixed order; value q PW + w's sum goes to
// t[q] of wave w.  Each round passes PW values through LDS, so all waves add (a
// tree over the waves left most of them idle: 600 cycles more of the 10000 of
// a workgroup at n = 1025 on MI355X).  Every thread of the workgroup (PW waves) calls it.
template <int N>
constexpr int NSHARE = (N + PW - 1) / PW;
template <int N>
__device__ __forceinline__ void waves_share(const double (&v)[N], int wave, int lane,
                                            double (&t)[NSHARE<N>])
{
    __shared__ double sh[PW][PW][RB];
#pragma unroll
    for (int q = 0; q < NSHARE<N>; ++q) {
        if (q > 0) __syncthreads();
#pragma unroll
        for (int k = 0; k < PW; ++k)
            if (q * PW + k < N) sh[k][wave][lane] = v[q * PW + k];
        __syncthreads();
        t[q] = 0.0;
        if (q * PW + wave < N) {
            double u[PW];
#pragma unroll
            for (int k = 0; k < PW; ++k) u[k] = sh[wave][k][lane];
#pragma unroll
            for (int h = PW / 2; h >= 1; h >>= 1)
#pragma unroll
                for (int k = 0; k < h; ++k) u[k] += u[k + h];
            t[q] = u[0];
        }
    }
}

// A wave's sums a for star i over records [R.j0, R.j1).
__device__ __forceinline__ void part64(const JRec64* __restrict__ jr, const JRange& R, int i,
                                       const I64& I, double (&a)[NACC], double eps2)
{
#pragma unroll
    for (int k = 0; k < NACC; ++k) a[k] = 0.0;
    if (R.w0 < R.w1) {
        run64<false, 0>(jr, R.j0, R.w0, i, I, a, eps2);
        run64<true, 0>(jr, R.w0, R.w1, i, I, a, eps2);
        run64<false, 0>(jr, R.w1, R.j1, i, I, a, eps2);
    } else {
        run64<false, 0>(jr, R.j0, R.j1, i, I, a, eps2);
    }
}

// Held to k_pair64's 7 waves per SIMD (72 VGPRs; 80 otherwise).
inline __global__ __launch_bounds__(PW * RB) __attribute__((amdgpu_waves_per_eu(7, 8)))
void k_pair64w(const JRec64* __restrict__ jr, const double* __restrict__ st,
               double* __restrict__ part, Phys P, int S, int nrow, int bid0)
{
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    int s, ig;
    const JRange R = j_part(bid0 + (int)blockIdx.x, S, nrow, wave, P.n, s, ig);
    const int n = P.n, li = ig * RB + lane + 1, i = li < n ? li : n - 1;
    const I64 I = load_i64(jr, st, P.cap, i, P.eps2);
    double a[NACC];
    part64(jr, R, i, I, a, P.eps2);
    double t[NSHARE<NACC>];
    waves_share(a, wave, lane, t);
    if (li < n) {
#pragma unroll
        for (int q = 0; q < NSHARE<NACC>; ++q)
            stream_out(t[q], &part[(size_t)(s * NACC + q * PW + wave) * P.cap + li]);
    }
}

// ---------------------------------------------------------------------
// force pair kernel, mixed: FP32 pair arithmetic on double-single
// positions, FP32 tile sums folded into Kahan-compensated FP32 totals, and
// the Newtonian term of the few pairs that can dominate a star's
// acceleration in FP64
// ---------------------------------------------------------------------
struct I32 {
    float xh, yh, zh, xl, yl, zl, gx, gy, gz, hx, hy, hz, D2e, rc2, dn2;
};

// Star i: its double-single position relative to its BH (particle b0; as
// in its mixed record, which is neutral if the star is close to the BH, so
// it is rebuilt from the FP64 record), velocity, |d_i|^2 and pair
// thresholds.
__device__ __forceinline__ I32 load_i32(const JRec64* __restrict__ j64,
                                        const Thr* __restrict__ thr,
                                        const double* __restrict__ st, int cap, int i, int b0,
                                        double eps2)
{
    const JRec64& r = j64[i];
    const double vx = st[3 * cap + i], vy = st[4 * cap + i], vz = st[5 * cap + i];
    const double D2 = r.D2;
    const Thr t = thr[i];
    double dx, dy, dz;
    {
#pragma clang fp contract(off)
        dx = r.x - st[b0];
        dy = r.y - st[cap + b0];
        dz = r.z - st[2 * cap + b0];
    }
    I32 I;
    I.xh = (float)dx; I.yh = (float)dy; I.zh = (float)dz;
    I.xl = (float)(dx - (double)I.xh);
    I.yl = (float)(dy - (double)I.yh);
    I.zl = (float)(dz - (double)I.zh);
    I.gx = (float)(4.0 * vx); I.gy = (float)(4.0 * vy); I.gz = (float)(4.0 * vz);
    I.hx = (float)(PN1_4OSQ15 * vx); I.hy = (float)(PN1_4OSQ15 * vy);
    I.hz = (float)(PN1_4OSQ15 * vz);
    I.D2e = (float)(D2 + eps2);
    I.rc2 = t.rc2;
    I.dn2 = t.dn2;
    return I;
}

// Folds the short-run FP32 Newtonian sums into their Kahan totals (total =
// sN - cN).
__device__ __forceinline__ void fold_newton(float (&a)[NACC32], float (&sN)[3], float (&cN)[3])
{
#pragma unroll
    for (int k = 0; k < 3; ++k) {
#pragma clang fp contract(off)
        const float y = a[A_NX + k] - cN[k];
        const float u = sN[k] + y;
        cN[k] = (u - sN[k]) - y;
        sN[k] = u;
        a[A_NX + k] = 0.0f;
    }
}

// u = fl(s + y), and its rounding error (Knuth's TwoSum, exact for any
// magnitudes) taken off the compensation c of a total kept as s - c.
__device__ __forceinline__ void two_sum_into(float s, float y, float& u, float& c)
{
#pragma clang fp contract(off)
    u = s + y;
    const float bv = u - s;
    const float av = u - bv;
    c -= (s - av) + (y - bv);
}

// Close pairs (R2e < rc2, not the self pair), taken when any lane of the
// wave has one; `close` selects the lanes.  A close pair's Newtonian term
// (m_j / mscale) w^3 r is evaluated in FP64 (rscale = 1 / mscale), from
// the mass of j's FP64 record and the double-single positions of j (its
// mixed record Js) and of the lane, and goes into the Kahan total; the
// FP32 term
// mw3 r that the caller adds next is cancelled exactly: the short-run sum
// is folded, then set to -p with p = fl(mw3 r), so the caller's
// fma(mw3, r, -p) leaves the exact product residual e = mw3 r - p, and
// T64 - e enters the total (as hi + lo floats: hi by TwoSum, lo into the
// compensation).  Every lane computes; the other lanes keep their sums.
// The branch around it is wave-uniform, so j and the record stream stay
// scalar.
__device__ __forceinline__ void close_pairs(bool close, const JRec64& J, const JRec32& Js,
                                            const I32& I, double eps2, double rscale, float mw3,
                                            float rx, float ry, float rz, float (&a)[NACC32],
                                            float (&sN)[3], float (&cN)[3])
{
#pragma clang fp contract(off)
    // the lane's position (double-single, relative to the BH: hi + lo is it
    // to 2^-48), made opaque here so that its FP64 form is built in this
    // rarely taken branch rather than hoisted out of the j loop and kept
    // live across it; j's from its mixed record, the same way
    float ph[3] = {I.xh, I.yh, I.zh}, pl[3] = {I.xl, I.yl, I.zl};
#pragma unroll
    for (int k = 0; k < 3; ++k) __asm__ volatile("" : "+v"(ph[k]), "+v"(pl[k]));
    const double dx = ((double)Js.xh + (double)Js.xl) - ((double)ph[0] + (double)pl[0]);
    const double dy = ((double)Js.yh + (double)Js.yl) - ((double)ph[1] + (double)pl[1]);
    const double dz = ((double)Js.zh + (double)Js.zl) - ((double)ph[2] + (double)pl[2]);
    const float jm32 = Js.m;
    const double R2 = __builtin_fma(dx, dx, __builtin_fma(dy, dy, __builtin_fma(dz, dz, eps2)));
    const double w = rsq64(R2);
    // in the record's mass units; none for a star taken out of the FP32 pass
    // (its mixed record, mass jm32, is neutral)
    const double mw3d = (jm32 != 0.0f ? J.m * rscale : 0.0) * (w * (w * w));
    const double d[3] = {dx, dy, dz};
    const float r[3] = {rx, ry, rz};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float p = mw3 * r[k];
        const float e = __builtin_fmaf(mw3, r[k], -p);
        const double D = mw3d * d[k] - (double)e;
        const float hi = (float)D;
        const float lo = (float)(D - (double)hi);
        // total = s - c; the short-run sum, then hi + lo, are added with
        // TwoSum, exact whatever the magnitudes (Kahan's update is exact
        // only while the running sum is the larger addend, and a star whose
        // terms cancel to a small |a| breaks that)
        float s1, c1 = cN[k];
        two_sum_into(sN[k], a[A_NX + k], s1, c1);
        float s2 = s1;
        two_sum_into(s1, hi, s2, c1);
        c1 -= lo;
        a[A_NX + k] = close ? -p : a[A_NX + k];
        sN[k] = close ? s2 : sN[k];
        cN[k] = close ? c1 : cN[k];
    }
}

// FP32 reciprocal square root of the pair kernels (RF: one Newton step,
// v_rsq_f32 ~1.6 ulp -> ~1 ulp).
template <bool RF>
__device__ __forceinline__ float rsq32(float R2e)
{
    float w = __builtin_amdgcn_rsqf(R2e);
    if (RF) {
        const float r = __builtin_fmaf(-(R2e * w), w, 1.0f);
        w = __builtin_fmaf(0.5f * w, r, w);
    }
    return w;
}

// One pair.  TS: also accumulate A_TS (the evaluations that refresh the
// stars' cancellation ratios).  EQ: every star of the cluster(s) has the
// same mass, so the record's mass m_j / mscale is 1 exactly (the self pair
// of the masked band keeps its zero mass) and m_j w is w.
template <bool MASK, bool RF, bool TS, bool EQ>
__device__ __forceinline__ void body32(const JRec32& J, const JRec64* __restrict__ j64, int j,
                                       int i, const I32& I, float (&a)[NACC32], float (&sN)[3],
                                       float (&cN)[3], float eps2, double eps2d, double rscale)
{
    float mj = J.m, MBj = J.MB, Qdx = J.Qdx, Qdy = J.Qdy, Qdz = J.Qdz;
    if (MASK) {
        const bool self = (j == i);
        mj = self ? 0.0f : mj;
        MBj = self ? 0.0f : MBj;
        Qdx = self ? 0.0f : Qdx;
        Qdy = self ? 0.0f : Qdy;
        Qdz = self ? 0.0f : Qdz;
    }
    // Separation from the hi parts of the positions; inside the lane's dn2
    // the lo parts are added, which gives the double-single separation
    // (x_hi,j - x_hi,i) + (x_lo,j - x_lo,i), so close pairs keep their digits.
    float rx = J.xh - I.xh, ry = J.yh - I.yh, rz = J.zh - I.zh;
    float R2e = __builtin_fmaf(rx, rx, __builtin_fmaf(ry, ry, __builtin_fmaf(rz, rz, eps2)));
    if (R2e < I.dn2) {
        rx += J.xl - I.xl;
        ry += J.yl - I.yl;
        rz += J.zl - I.zl;
        R2e = __builtin_fmaf(rx, rx, __builtin_fmaf(ry, ry, __builtin_fmaf(rz, rz, eps2)));
        // close pairs (dn2 >= rc2, so they are all in this branch): their
        // FP32 mw3 is formed here as below, bit for bit
        const bool close = R2e < I.rc2 && (!MASK || j != i);
        if (__builtin_amdgcn_ballot_w64(close)) {
            const float wc = rsq32<RF>(R2e);
            const float mw3c = (EQ && !MASK ? wc : mj * wc) * (wc * wc);
            close_pairs(close, j64[j], J, I, eps2d, rscale, mw3c, rx, ry, rz, a, sN, cN);
        }
    }
    const float w = rsq32<RF>(R2e);
    const float w2 = w * w;
    constexpr bool UNIT = EQ && !MASK;
    const float mw = UNIT ? w : mj * w;
    const float mw3 = mw * w2;
    a[A_PHI] += mw;
    a[A_W3] += mw3;
    if (TS) a[A_TS] = UNIT ? a[A_TS] + w2 : __builtin_fmaf(mw, w, a[A_TS]);
    a[A_TX] = __builtin_fmaf(w, Qdx, a[A_TX]);
    a[A_TY] = __builtin_fmaf(w, Qdy, a[A_TY]);
    a[A_TZ] = __builtin_fmaf(w, Qdz, a[A_TZ]);
    const float t = R2e - I.D2e;
    a[A_ZE] = __builtin_fmaf(MBj, t, a[A_ZE]);
    const float sr = __builtin_fmaf(J.sx, rx, __builtin_fmaf(J.sy, ry, J.sz * rz));
    // the bracket starts from (s_j.r w)^2 + A_j: one record operand per
    // instruction (gfx950 reads one scalar register per VALU op), no copy
    const float tv = sr * w;
    float br = __builtin_fmaf(tv, tv, J.A);
    br = __builtin_fmaf(J.B, t, br);
    br = __builtin_fmaf(I.hx, J.sx, __builtin_fmaf(I.hy, J.sy, __builtin_fmaf(I.hz, J.sz, br)));
    const float Kr = mw3 * br;
    a[A_RX] = __builtin_fmaf(Kr, rx, a[A_RX]);
    a[A_RY] = __builtin_fmaf(Kr, ry, a[A_RY]);
    a[A_RZ] = __builtin_fmaf(Kr, rz, a[A_RZ]);
    const float gr = __builtin_fmaf(I.gx, rx, __builtin_fmaf(I.gy, ry, I.gz * rz));
    const float Ku = mw3 * __builtin_fmaf((float)-PN1_SQ6, sr, gr);
    a[A_UX] = __builtin_fmaf(Ku, J.sx, a[A_UX]);
    a[A_UY] = __builtin_fmaf(Ku, J.sy, a[A_UY]);
    a[A_UZ] = __builtin_fmaf(Ku, J.sz, a[A_UZ]);
    a[A_KS] += Ku;
    a[A_NX] = __builtin_fmaf(mw3, rx, a[A_NX]);
    a[A_NY] = __builtin_fmaf(mw3, ry, a[A_NY]);
    a[A_NZ] = __builtin_fmaf(mw3, rz, a[A_NZ]);
}

// Mixed-form j loop: PP bit 0 clear: one body at a time; set: two bodies
// per iteration, records two ahead (as run64).
// One j-record with a single 64-byte scalar load (one wait per pair instead
// of one per group of fields the body reaches).
typedef float f32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ JRec32 load_rec(const JRec32* __restrict__ p)
{
    const f32x16 v = *reinterpret_cast<const f32x16*>(p);
    JRec32 r;
    r.xh = v[0]; r.yh = v[1]; r.zh = v[2];
    r.xl = v[3]; r.yl = v[4]; r.zl = v[5];
    r.sx = v[6]; r.sy = v[7]; r.sz = v[8];
    r.m = v[9]; r.A = v[10]; r.B = v[11]; r.MB = v[12];
    r.Qdx = v[13]; r.Qdy = v[14]; r.Qdz = v[15];
    return r;
}

// A wave-uniform pair counter folds the Newtonian sums into Kahan totals
// every `tile` pairs without restarting the record stream.
template <bool MASK, int PP, bool TS, bool EQ>
__device__ __forceinline__ void run32(const JRec32* __restrict__ jr,
                                      const JRec64* __restrict__ j64, int j0, int j1, int i,
                                      const I32& I, float (&a)[NACC32], float eps2, double eps2d,
                                      double rscale, float (&sN)[3], float (&cN)[3], int tile,
                                      int& cnt)
{
    constexpr bool RF = (PP & 2) != 0;
    if ((PP & 1) == 0) {
        for (int j = j0; j < j1; ++j) {
            body32<MASK, RF, TS, EQ>(load_rec(jr + j), j64, j, i, I, a, sN, cN, eps2, eps2d,
                                     rscale);
            if (++cnt >= tile) {
                cnt = 0;
                fold_newton(a, sN, cN);
            }
        }
        return;
    }
    if (j0 >= j1) return;
    JRec32 ra = jr[j0];
    int j = j0;
    for (; j + 1 < j1; j += 2) {
        const JRec32 rb = jr[j + 1];
        body32<MASK, RF, TS, EQ>(ra, j64, j, i, I, a, sN, cN, eps2, eps2d, rscale);
        ra = jr[j + 2];
        body32<MASK, RF, TS, EQ>(rb, j64, j + 1, i, I, a, sN, cN, eps2, eps2d, rscale);
        cnt += 2;
        if (cnt >= tile) {
            cnt = 0;
            fold_newton(a, sN, cN);
        }
    }
    if (j < j1) {
        body32<MASK, RF, TS, EQ>(ra, j64, j, i, I, a, sN, cN, eps2, eps2d, rscale);
        ++cnt;
    }
}


// The Newtonian sums are Kahan-compensated every `tile` pairs (at least
// 2; 64 by default): they carry the stars' accelerations, and with the
// close pairs taken out of the FP32 run sums, a run holds no term larger
// than PN1_CLOSE_KAPPA |a|.  The other sums enter scaled by 1/c^2 (or, for the
// BH, beside its FP64 Newtonian term) and accumulate in plain FP32 over
// the whole chunk.
// The one-record form is held to 8 waves per SIMD: under the max-ILP
// scheduler (pn1_pair32.hip) it would otherwise take 65 VGPRs.
template <int PP, bool TS, bool EQ>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu((PP & 1) ? 1 : 8, 8)))
void k_pair32(const JRec32* __restrict__ jr, const JRec64* __restrict__ j64,
              const Thr* __restrict__ thr, const double* __restrict__ st,
              float* __restrict__ part, Phys P, int S, int nIblk, int ib0, int tile)
{
    int s, ib;
    map_block(blockIdx.x, S, nIblk, s, ib);
    if (ib >= nIblk) return;
    ib += ib0;
    const int n = P.n;
    const int li = ib * WG + threadIdx.x + 1;
    const int i = li < n ? li : n - 1;
    const I32 I = load_i32(j64, thr, st, P.cap, i, 0, P.eps2);
    const JRange R = j_range(s, S, n, ib);
    const float eps2 = P.eps2f;
    const double eps2d = P.eps2, rscale = 1.0 / P.mmax;
    float a[NACC32], sumN[3], cmpN[3];
#pragma unroll
    for (int k = 0; k < NACC32; ++k) a[k] = 0.0f;
#pragma unroll
    for (int k = 0; k < 3; ++k) sumN[k] = cmpN[k] = 0.0f;
    int cnt = 0;
    if (R.w0 < R.w1) {
        run32<false, PP, TS, EQ>(jr, j64, R.j0, R.w0, i, I, a, eps2, eps2d, rscale, sumN, cmpN, tile, cnt);
        run32<true, PP, TS, EQ>(jr, j64, R.w0, R.w1, i, I, a, eps2, eps2d, rscale, sumN, cmpN, tile, cnt);
        run32<false, PP, TS, EQ>(jr, j64, R.w1, R.j1, i, I, a, eps2, eps2d, rscale, sumN, cmpN, tile, cnt);
    } else {
        run32<false, PP, TS, EQ>(jr, j64, R.j0, R.j1, i, I, a, eps2, eps2d, rscale, sumN, cmpN, tile, cnt);
    }
    fold_newton(a, sumN, cmpN);
    if (li < n) {
        // [s][MROWS][cap]: the sums, then the Newtonian compensations
        const size_t cap = (size_t)P.cap;
        float* ps = part + (size_t)s * MROWS * cap + li;
#pragma unroll
        for (int k = 0; k < NACC32; ++k)
            if (TS || k != A_TS) stream_out(k <= A_NZ ? sumN[k] : a[k], &ps[k * cap]);
#pragma unroll
        for (int k = 0; k < 3; ++k) stream_out(cmpN[k], &ps[(NACC32 + k) * cap]);
    }
}

// The same pairs in workgroups of four i-waves x four consecutive j
// chunks (1024 threads): wave w takes the i-stars of i-wave w % 4 of block
// ib against chunk 4 s4 + w / 4 of the split in S chunks, so every wave
// does what it does in k_pair32 (and its FP32 sums are the same bits), but
// the four chunk sums of each star are combined in LDS and written as one
// partial of the split in S / 4 chunks: a quarter of k_pair32's partial-sum
// traffic.  The combination is in FP64: the Newtonian totals s - c are
// written back as a hi/lo float pair (s = hi, c = -lo, so that k_fin's
// s - c is the FP64 total to ~2^-48), the other sums rounded once to FP32.
constexpr int QSUB = 4;
constexpr int WGQ = QSUB * WG;
template <int PP, bool TS, bool EQ>
__global__ __launch_bounds__(WGQ) __attribute__((amdgpu_waves_per_eu(8, 8)))
void k_pair32q(const JRec32* __restrict__ jr, const JRec64* __restrict__ j64,
               const Thr* __restrict__ thr, const double* __restrict__ st,
               float* __restrict__ part, Phys P, int S, int nIblk, int ib0, int tile)
{
    __shared__ float red[QSUB - 1][MROWS][WG];
    const int S4 = S / QSUB;
    int s4, ib;
    map_block(blockIdx.x, S4, s4, ib);
    if (ib >= nIblk) return;                  // the whole workgroup
    ib += ib0;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int iw = wave & 3, sub = wave >> 2, lane = threadIdx.x & 63;
    const int n = P.n;
    const int li = ib * WG + iw * 64 + lane + 1;
    const int i = li < n ? li : n - 1;
    const I32 I = load_i32(j64, thr, st, P.cap, i, 0, P.eps2);
    // chunk 4 s4 + sub of the S-chunk split (k_pair32's bounds), and the
    // self window of this wave's 64 stars
    JRange R = j_range(s4 * QSUB + sub, S, n, ib);
    {
        const int wb = ib * WG + iw * 64 + 1;
        R.w0 = max(R.j0, wb);
        R.w1 = min(R.j1, wb + 64);
    }
    const float eps2 = P.eps2f;
    const double eps2d = P.eps2, rscale = 1.0 / P.mmax;
    float a[NACC32], sumN[3], cmpN[3];
#pragma unroll
    for (int k = 0; k < NACC32; ++k) a[k] = 0.0f;
#pragma unroll
    for (int k = 0; k < 3; ++k) sumN[k] = cmpN[k] = 0.0f;
    int cnt = 0;
    if (R.w0 < R.w1) {
        run32<false, PP, TS, EQ>(jr, j64, R.j0, R.w0, i, I, a, eps2, eps2d, rscale, sumN, cmpN, tile, cnt);
        run32<true, PP, TS, EQ>(jr, j64, R.w0, R.w1, i, I, a, eps2, eps2d, rscale, sumN, cmpN, tile, cnt);
        run32<false, PP, TS, EQ>(jr, j64, R.w1, R.j1, i, I, a, eps2, eps2d, rscale, sumN, cmpN, tile, cnt);
    } else if (R.j0 < R.j1) {
        run32<false, PP, TS, EQ>(jr, j64, R.j0, R.j1, i, I, a, eps2, eps2d, rscale, sumN, cmpN, tile, cnt);
    }
    fold_newton(a, sumN, cmpN);
    const int col = iw * 64 + lane;
    if (sub > 0) {
#pragma unroll
        for (int k = 0; k < NACC32; ++k)
            if (TS || k != A_TS) red[sub - 1][k][col] = k <= A_NZ ? sumN[k] : a[k];
#pragma unroll
        for (int k = 0; k < 3; ++k) red[sub - 1][NACC32 + k][col] = cmpN[k];
    }
    __syncthreads();
    if (sub == 0 && li < n) {
        const size_t cap = (size_t)P.cap;
        float* ps = part + (size_t)s4 * MROWS * cap + li;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            double t = (double)sumN[k] - (double)cmpN[k];
#pragma unroll
            for (int q = 0; q < QSUB - 1; ++q)
                t += (double)red[q][k][col] - (double)red[q][NACC32 + k][col];
            const float hi = (float)t;
            stream_out(hi, &ps[k * cap]);
            stream_out(-(float)(t - (double)hi), &ps[(NACC32 + k) * cap]);
        }
#pragma unroll
        for (int k = A_NZ + 1; k < NACC32; ++k) {
            if (!TS && k == A_TS) continue;
            double t = (double)a[k];
#pragma unroll
            for (int q = 0; q < QSUB - 1; ++q) t += (double)red[q][k][col];
            stream_out((float)t, &ps[k * cap]);
        }
    }
}

// A wave's sums for star i over records [R.j0, R.j1): a, and the Newtonian
// ones as sumN - cmpN (rscale: 1 / the records' mass scale).
template <bool TS, bool EQ>
__device__ __forceinline__ void part32(const JRec32* __restrict__ jr,
                                       const JRec64* __restrict__ j64, const JRange R, int i,
                                       const I32& I, float eps2, double eps2d, double rscale,
                                       int tile, float (&a)[NACC32], float (&sumN)[3],
                                       float (&cmpN)[3])
{
#pragma unroll
    for (int k = 0; k < NACC32; ++k) a[k] = 0.0f;
#pragma unroll
    for (int k = 0; k < 3; ++k) sumN[k] = cmpN[k] = 0.0f;
    int cnt = 0;
    if (R.w0 < R.w1) {
        run32<false, 0, TS, EQ>(jr, j64, R.j0, R.w0, i, I, a, eps2, eps2d, rscale, sumN, cmpN, tile, cnt);
        run32<true, 0, TS, EQ>(jr, j64, R.w0, R.w1, i, I, a, eps2, eps2d, rscale, sumN, cmpN, tile, cnt);
        run32<false, 0, TS, EQ>(jr, j64, R.w1, R.j1, i, I, a, eps2, eps2d, rscale, sumN, cmpN, tile, cnt);
    } else {
        run32<false, 0, TS, EQ>(jr, j64, R.j0, R.j1, i, I, a, eps2, eps2d, rscale, sumN, cmpN, tile, cnt);
    }
    fold_newton(a, sumN, cmpN);
}

// The sums of the workgroup's waves, added in FP64, as partials (rows of
// `stride` floats from ps): the Newtonian totals as a hi/lo float pair (s = hi,
// c = -lo, so that k_fin's s - c is the FP64 total to ~2^-48), the others
// rounded once to FP32.  ok: the lane has a star.
template <bool TS>
__device__ __forceinline__ void put_part32(const float (&a)[NACC32], const float (&sumN)[3],
                                           const float (&cmpN)[3], int wave, int lane, bool ok,
                                           float* __restrict__ ps, size_t stride)
{
    constexpr int NV = TS ? NACC32 : NACC;
    double v[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k)
        v[k] = k <= A_NZ ? (double)sumN[k] - (double)cmpN[k] : (double)a[k];
    double t[NSHARE<NV>];
    waves_share(v, wave, lane, t);
    if (ok) {
#pragma unroll
        for (int q = 0; q < NSHARE<NV>; ++q) {
            const int k = q * PW + wave;
            if (k >= NV) break;
            const float hi = (float)t[q];
            stream_out(hi, &ps[k * stride]);
            if (k <= A_NZ) stream_out(-(float)(t[q] - (double)hi), &ps[(NACC32 + k) * stride]);
        }
    }
}

// Hard stars (PN1_HARD_K) of the row kernels: the FP64 sums of a row's first
// HSLOT of them over chunk [j0, j1), one record per lane, NACC sums and sum m_j
// w^2 each, to out + slot HCHUNK (NACC + 1); k_fin adds the chunks' (hard_sum).
// By k_fin's one workgroup for the row (rare_rows) a star takes 15 us at n =
// 10241 on MI355X while the rest of the chip waits; here its chunks run beside
// other rows' work.  Not inlined, and held to the pair kernel's registers: the
// call is rare.  With one hard star, evaluation: n = 10241, 135 -> 122 us, n =
// 12289, 197 -> 162, n = 16385, 271 -> 239.  Every thread of the workgroup calls
// it.
constexpr int HSLOT = 2, HCHUNK = TLONG + TSHORT;
constexpr int HROWS = 4096, EHROWS = 16384;  // rows with room for them (EHROWS: of an ensemble)
__attribute__((noinline)) __device__ void
hard_part(const JRec64* __restrict__ jr, const double* __restrict__ st, int cap, double eps2,
          int i0, unsigned long long hm, int j0, int j1, double* __restrict__ out)
{
    __shared__ double wsum[NACC + 1][PW];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (int slot = 0; slot < HSLOT && hm; ++slot) {
        const int i = i0 + __builtin_ctzll(hm);
        hm &= hm - 1;
        const I64 I = load_i64(jr, st, cap, i, eps2);
        double a[NACC], ts = 0.0;
#pragma unroll
        for (int k = 0; k < NACC; ++k) a[k] = 0.0;
        for (int j = j0 + (int)threadIdx.x; j < j1; j += PW * RB) {
            const JRec64& J = jr[j];
            body64<true>(J, j, i, I, a, eps2);
            if (j != i) {
                const double rx = J.x - I.x, ry = J.y - I.y, rz = J.z - I.z;
                ts += J.m / (rx * rx + ry * ry + rz * rz + eps2);
            }
        }
        const double u = wave_sums16(a), w = wave_sum(ts);
        if ((lane & 3) == 0) wsum[lane >> 2][wid] = u;
        if (lane == 0) wsum[NACC][wid] = w;
        __syncthreads();
        if (threadIdx.x <= NACC) {
            double t = 0.0;
#pragma unroll
            for (int k = 0; k < PW; ++k) t += wsum[threadIdx.x][k];
            out[(size_t)slot * HCHUNK * (NACC + 1) + threadIdx.x] = t;
        }
        __syncthreads();
    }
}

// A hard star's sums over its S chunks hp: lane k <= NACC gets value k.
__device__ __forceinline__ double hard_sum(const double* __restrict__ hp, int S)
{
    constexpr int N = NACC + 1;
    const int lane = threadIdx.x & 63, v = lane % N, g = lane / N;
    double t = 0.0;
    if (g < 3) {
#pragma unroll 8
        for (int s = g; s < S; s += 3) t += hp[s * N + v];
    }
    const double b = __shfl(t, min(lane + N, 63), 64), c = __shfl(t, min(lane + 2 * N, 63), 64);
    return (t + b) + c;
}

// k_pair64w's form of the mixed kernel.
template <bool TS, bool EQ>
__global__ __launch_bounds__(PW * RB) __attribute__((amdgpu_waves_per_eu(8, 8)))
void k_pair32w(const JRec32* __restrict__ jr, const JRec64* __restrict__ j64,
               const Thr* __restrict__ thr, const double* __restrict__ st,
               float* __restrict__ part, Phys P, int S, int nrow, int bid0, int tile,
               const unsigned long long* __restrict__ hmask, double* __restrict__ hpart)
{
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    int s, ig;
    const JRange R = j_part(bid0 + (int)blockIdx.x, S, nrow, wave, P.n, s, ig);
    const int n = P.n, li = ig * RB + lane + 1, i = li < n ? li : n - 1;
    const I32 I = load_i32(j64, thr, st, P.cap, i, 0, P.eps2);
    float a[NACC32], sumN[3], cmpN[3];
    part32<TS, EQ>(jr, j64, R, i, I, P.eps2f, P.eps2, 1.0 / P.mmax, tile, a, sumN, cmpN);
    put_part32<TS>(a, sumN, cmpN, wave, lane, li < n, part + (size_t)s * MROWS * P.cap + li,
                   (size_t)P.cap);
    if (hpart) {
        const unsigned long long hm = hmask[ig];
        if (hm) {
            // the whole chunk: from wave 0's part to the last wave's
            int s0, g0;
            const JRange A = j_part(bid0 + (int)blockIdx.x, S, nrow, 0, n, s0, g0);
            const JRange B = j_part(bid0 + (int)blockIdx.x, S, nrow, PW - 1, n, s0, g0);
            hard_part(j64, st, P.cap, P.eps2, 1 + ig * RB, hm, A.j0, B.j1,
                      hpart + ((size_t)ig * HSLOT * HCHUNK + s) * (NACC + 1));
        }
    }
}

// ---------------------------------------------------------------------
// k_fin: star accelerations, stage update, BH, the next evaluation's prep
// ---------------------------------------------------------------------
// The local stars [first, first + 64 nrow) of a cluster (BH at off, nst
// stars) whose sums need more than the FP32 pass gave, mixed form: x at the
// star's index gets, [NACC + 1][cap] (the NACC sums and sum m_j w^2, from the
// FP64 form's body),
//   a hard star (hmask of the rows, see PN1_HARD_K; but for each row's first
//     `skip`, which hard_part has done): its whole row over the
//     cluster's records (BH-close stars included, with their full records),
//     reduced over the workgroup's FWG lanes in a fixed order;
//   any other star: its pairs with the nf BH-close stars (flist, see
//     PN1_FLAG_ETA), if there are any.
// Row r's star part runs in wave r (wave 0 if nrow is 1).  Every thread of
// the workgroup calls it.  A call, not inlined, ahead of k_fin's own work: it
// is rare, and inlined its registers would halve k_fin's occupancy.
__attribute__((noinline)) __device__ void rare_rows(const JRec64* __restrict__ jr,
                                                    const double* __restrict__ st, int cap,
                                                    double eps2, int off, int nst, int first,
                                                    int nrow,
                                                    const unsigned long long* __restrict__ hmask,
                                                    int shift, unsigned long long width,
                                                    int nall, int skip,
                                                    const int* __restrict__ flist, int nf,
                                                    double* __restrict__ x)
{
    __shared__ double wsum[NACC + 1][FG];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    double a[NACC], ts;
    auto pair = [&](int j, int i, const I64& I) {
        const JRec64& J = jr[j];
        body64<true>(J, j, i, I, a, eps2);
        if (j != i) {
            const double rx = J.x - I.x, ry = J.y - I.y, rz = J.z - I.z;
            ts += J.m / (rx * rx + ry * ry + rz * rz + eps2);
        }
    };
    if (nf > 0 && wid < nrow && first + (int)threadIdx.x < nst) {
        const int i = off + 1 + first + (int)threadIdx.x;
        const I64 I = load_i64(jr, st, cap, i, eps2);
        ts = 0.0;
#pragma unroll
        for (int k = 0; k < NACC; ++k) a[k] = 0.0;
        for (int f = 0; f < nf; ++f) pair(flist[f], i, I);
#pragma unroll
        for (int k = 0; k < NACC; ++k) x[(size_t)k * cap + i] = a[k];
        x[(size_t)NACC * cap + i] = ts;
    }
    for (int r = 0; r < nrow && first + r * RB < nst; ++r) {
        unsigned long long hm = hmask[r];
        for (int k = 0; k < skip; ++k) hm &= hm - 1;      // those of hard_part
        hm = (hm >> shift) & width;
        while (hm) {
            const int h = r * RB + __builtin_ctzll(hm), i = off + 1 + first + h;
            hm &= hm - 1;
            const I64 I = load_i64(jr, st, cap, i, eps2);
            ts = 0.0;
#pragma unroll
            for (int k = 0; k < NACC; ++k) a[k] = 0.0;
            for (int j = off + 1 + (int)threadIdx.x; j <= off + nall; j += FWG) pair(j, i, I);
#pragma unroll
            for (int k = 0; k <= NACC; ++k) {
                const double t = wave_sum(k < NACC ? a[k] : ts);
                if (lane == 0) wsum[k][wid] = t;
            }
            __syncthreads();
            if ((int)threadIdx.x == h)
#pragma unroll
                for (int k = 0; k <= NACC; ++k) {
                    double t = 0.0;
                    for (int w = 0; w < FG; ++w) t += wsum[k][w];
                    x[(size_t)k * cap + i] = t;
                }
            __syncthreads();
        }
    }
}

// Sum of the S chunk partials of one row of stars, by G waves (G = 1 or FG):
// wave g adds chunks g, g + G, ... of the lane's star, and the waves' sums
// are added pairwise in a fixed order; the result is in wave 0 of the G.
// `part` points at the cluster's partial area, `stride` is its per-sum
// stride and `idx` the star's index in it (any valid one for a lane without
// a star).  FP64: [S][NACC][stride]; mixed: [S][MROWS][stride] floats (the
// NACC32 sums, then the Newtonian Kahan compensations), whose sums built
// from the record's mass m_j / mscale are scaled back by mscale; A[NACC] is
// the mixed form's A_TS sum (TS: the stages whose pair kernels write it).
// Two chunks' loads are in flight at once: a partial comes from another XCD,
// 1.1 us away, and few waves run here.
template <int MODE, bool TS>
struct Chunk {
    static constexpr int NV = MODE == 1 && TS ? NACC + 1 : NACC;
    double L64[MODE == 0 ? NV : 1];
    float L32[MODE == 1 ? NV : 1], C[MODE == 1 ? 3 : 1];
    __device__ __forceinline__ void load(const void* __restrict__ part, int s, size_t stride,
                                         size_t idx)
    {
        if (MODE == 0) {
            const double* pp = (const double*)part + (size_t)s * NACC * stride + idx;
#pragma unroll
            for (int k = 0; k < NV; ++k) L64[k] = __builtin_nontemporal_load(&pp[k * stride]);
        } else {
            const float* ps = (const float*)part + (size_t)s * MROWS * stride + idx;
#pragma unroll
            for (int k = 0; k < NV; ++k) L32[k] = __builtin_nontemporal_load(&ps[k * stride]);
#pragma unroll
            for (int k = 0; k < 3; ++k)
                C[k] = __builtin_nontemporal_load(&ps[(NACC32 + k) * stride]);
        }
    }
    __device__ __forceinline__ void add(double (&A)[NACC + 1]) const
    {
#pragma unroll
        for (int k = 0; k < NV; ++k) A[k] += MODE == 0 ? L64[k] : (double)L32[k];
        if (MODE == 1)
#pragma unroll
            for (int k = 0; k < 3; ++k) A[A_NX + k] -= (double)C[k];
    }
};

template <int MODE, bool TS, int G>
__device__ __forceinline__ void gather_row(const void* __restrict__ part, int S, size_t stride,
                                           size_t idx, double mscale, double (&A)[NACC + 1])
{
    constexpr int NV = Chunk<MODE, TS>::NV;
    const int lane = threadIdx.x & 63;
    const int g = G == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
#pragma unroll
    for (int k = 0; k <= NACC; ++k) A[k] = 0.0;
    Chunk<MODE, TS> c0, c1;
    int s = g;
    if (G > 1)
        for (; s + G < S; s += 2 * G) {
            c0.load(part, s, stride, idx);
            c1.load(part, s + G, stride, idx);
            __builtin_amdgcn_sched_barrier(0);       // all of their loads in flight
            c0.add(A);
            c1.add(A);
        }
    for (; s < S; s += G) {
        c0.load(part, s, stride, idx);
        __builtin_amdgcn_sched_barrier(0);
        c0.add(A);
    }
    if (MODE == 1)
#pragma unroll
        for (int k = 0; k < NV; ++k)
            if (k <= A_UZ || k == A_KS || k == A_PHI || k == A_W3 || k == A_TS) A[k] *= mscale;
    if (G > 1) {
        __shared__ double sum[G > 1 ? NV : 1][RB];
        double v[NV], t[NSHARE<NV>];
#pragma unroll
        for (int k = 0; k < NV; ++k) v[k] = A[k];
        waves_share(v, g, lane, t);
#pragma unroll
        for (int q = 0; q < NSHARE<NV>; ++q)
            if (q * PW + g < NV) sum[G > 1 ? q * PW + g : 0][lane] = t[q];
        __syncthreads();
        if (g == 0)
#pragma unroll
            for (int k = 0; k < NV; ++k) A[k] = sum[G > 1 ? k : 0][lane];
    }
}

// The same for 16 stars by the FG waves of a workgroup: lane l has star l % 16,
// and its quarter of wave w adds chunks 4 w + l / 16, ... + 4 FG, ...; the
// sums over chunks are in every quarter of wave 0.
template <int MODE, bool TS>
__device__ __forceinline__ void gather_sub(const void* __restrict__ part, int S, size_t stride,
                                           size_t idx, double mscale, double (&A)[NACC + 1])
{
    constexpr int NV = Chunk<MODE, TS>::NV, RS = 16;
    __shared__ double sh[FG][NV][RS], sum[NV][RS];
    const int lane = threadIdx.x & 63, ls = lane % RS;
    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nw = min(FG, (S + 3) / 4);             // waves with a chunk
#pragma unroll
    for (int k = 0; k <= NACC; ++k) A[k] = 0.0;
    if (wid < nw) {
        for (int s = wid * 4 + lane / RS; s < S; s += 4 * FG) {
            Chunk<MODE, TS> c;
            c.load(part, s, stride, idx);
            __builtin_amdgcn_sched_barrier(0);
            c.add(A);
        }
        // quarter q of the wave: values 8 (q / 2) + 4 (q % 2) + 0 .. 3
        double a[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) a[k] = swap_sum<32>(A[k], A[8 + k]);
        const int v0 = 8 * (lane >> 5) + 4 * ((lane >> 4) & 1);
#pragma unroll
        for (int k = 0; k < 4; ++k) sh[wid][v0 + k][ls] = swap_sum<16>(a[k], a[4 + k]);
        if (NV > NACC) {
            double t = A[NACC];
            t += __shfl_xor(t, 32, 64);
            t += __shfl_xor(t, 16, 64);
            if (lane < RS) sh[wid][NV - 1][ls] = t;
        }
    }
    __syncthreads();
    if (threadIdx.x < NV * RS) {
        const int k = threadIdx.x / RS;
        double t = sh[0][k][ls];
        for (int w = 1; w < nw; ++w) t += sh[w][k][ls];
        if (MODE == 1)
            if (k <= A_UZ || k == A_KS || k == A_PHI || k == A_W3 || k == A_TS) t *= mscale;
        sum[k][ls] = t;
    }
    __syncthreads();
    if (wid == 0)
#pragma unroll
        for (int k = 0; k < NV; ++k) A[k] = sum[k][ls];
}

// Mixed form: the star's cancellation ratio for the next evaluation's
// thresholds, sum m_j w^2 / |a| (NaN for a = 0, which counts as hard).
__device__ __forceinline__ float cancel_ratio(double ts, const double (&a)[3])
{
    return (float)(ts * rsq64(a[0] * a[0] + a[1] * a[1] + a[2] * a[2]));
}

// Run constants shared by the O(n) passes of one cluster.
struct FinC {
    double m0, eps, eps2, ws, lam, dt;
};

// Star p (BH of its cluster at x0) of mass mp in state st, with |d|^2 = D2 and
// e from its record: its acceleration
// from its pair sums S_ and the cluster's separable sums gs, the stage update
// (nx, nv: the state of the driver's next force call), and its share cb of
// the BH's 1PN acceleration (a1 + a1c).
template <int STAGE>
__device__ __forceinline__ void fin_star(const StageIn& st, const double (&x0)[3], double mp,
                                         double D2, double e,
                                         double* X, double* Y, double* H1, double* H2, int cap,
                                         int p, const double (&S_)[NACC + 1],
                                         const double (&gs)[NGS], const FinC& C,
                                         double* __restrict__ acc, double (&cb)[3],
                                         double (&a)[3], double (&nx)[3], double (&nv)[3])
{
    const double m0 = C.m0, eps2 = C.eps2;
    const double (&x)[3] = st.x, (&v)[3] = st.v;
    const double d[3] = {x[0] - x0[0], x[1] - x0[1], x[2] - x0[2]};
    const double E3 = e * e * e, q = mp * E3;
    const double G1 = gs[G_G1];
    const double M1[3] = {gs[G_M1X], gs[G_M1Y], gs[G_M1Z]};
    const double Pm[3] = {gs[G_PX], gs[G_PY], gs[G_PZ]};
    const double V2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
    const double vd = v[0] * d[0] + v[1] * d[1] + v[2] * d[2];

    // ---- star i: Newton + B + S + sum over j != i of the ac pair term
    const double Pp[3] = {Pm[0] - mp * v[0], Pm[1] - mp * v[1], Pm[2] - mp * v[2]};
    const double vP = v[0] * Pp[0] + v[1] * Pp[1] + v[2] * Pp[2];
    const double Pd = Pp[0] * d[0] + Pp[1] * d[1] + Pp[2] * d[2];
    const double c1 = -m0 * E3 * (4.0 * S_[A_PHI] + 1.25 * (G1 - mp * e)) + E3 * S_[A_ZE];
    const double cB = 4.0 * m0 * e - V2;   // also the i-only part of the K_r bracket
    const double cS = 5.0 * m0 * mp * e * e * e * e - 4.0 * mp * E3 * V2;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double newton = S_[A_NX + k] - m0 * E3 * d[k];
        const double B = -m0 * E3 * (d[k] * cB + 4.0 * vd * v[k]);
        const double Sg = cS * d[k] + 7.0 * mp * E3 * vd * v[k];
        const double t4 = E3 * (4.0 * vP * d[k] - 3.0 * Pd * v[k] - 4.0 * vd * Pp[k]);
        const double ru = S_[A_UX + k] * PN1_ISQ15 - v[k] * S_[A_KS];
        const double t3 = S_[A_TX + k] - 3.5 * m0 * e * (M1[k] - q * d[k]);
        const double rr = S_[A_RX + k] + cB * S_[A_NX + k];
        const double pn = B + Sg + rr + ru + c1 * d[k] + t3 + t4;
        a[k] = newton + C.lam * pn;
        acc[(size_t)k * cap + p] = a[k];
    }

    // ---- this star's share of the BH's 1PN acceleration: a1 + a1c
    // the j = i bracket of the a1c pair term in the reference's operation
    // order (Limit-sticky9.c:139-140 at |r|^2 = 0)
    double self_br;
    {
#pragma clang fp contract(off)
        const double ws = C.ws;
        self_br = 4.0 * e + 1.25 * ws - 0.25 * D2 / eps2 * ws + 0.25 * D2 / eps2 * ws;
    }
    const double vP0 = v[0] * Pm[0] + v[1] * Pm[1] + v[2] * Pm[2];
    const double Pd0 = Pm[0] * d[0] + Pm[1] * d[1] + Pm[2] * d[2];
    const double mE3 = mp * E3;
    const double cA1 = mE3 * (5.0 * m0 * e - 2.0 * V2 + 1.5 * vd * vd / D2);
    const double cC0 = 4.0 * mp * mp * e * e * e * e;
    // xi_i = sum' m_j w^3 (D2_i - D2_j) = -2 d_i.N - phi + eps^2 W3
    const double xi = -2.0 * (d[0] * S_[A_NX] + d[1] * S_[A_NY] + d[2] * S_[A_NZ])
                      - S_[A_PHI] + eps2 * S_[A_W3];
    const double cC2 = mE3 * (4.0 * (G1 - mp * e) + 1.25 * S_[A_PHI] + 0.25 * xi
                              + mp * self_br);
    const double cQ2 = mp * mp * E3 * (4.0 * e + 1.25 * C.eps);
    const double vm = mE3 / m0, vm2 = mp * vm;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double A1 = cA1 * d[k] + 3.0 * mE3 * vd * v[k];
        const double C2 = cC2 * d[k] - 3.5 * e * mp * S_[A_NX + k]
                          - vm * (4.0 * vP0 * d[k] - 3.0 * vd * Pm[k] - 4.0 * Pd0 * v[k]);
        const double Q2 = cQ2 * d[k] - vm2 * (4.0 * V2 * d[k] - 7.0 * vd * v[k]);
        cb[k] = A1 + cC0 * d[k] + C2 + Q2;
    }
#pragma unroll
    for (int k = 0; k < 3; ++k)
        stage_update<STAGE>(p, cap, st, k, k, a[k], X, Y, H1, H2, C.dt, nx[k], nv[k]);
}

__device__ __forceinline__ FinC fin_consts(const Phys& P, double m0)
{
    FinC C;
    C.m0 = m0;
    C.eps = P.eps;
    C.eps2 = P.eps2;
    C.ws = P.ws;
    C.lam = P.lam;
    C.dt = P.dt;
    return C;
}

// What k_fin works on besides the partial sums.  kr (mixed form): each
// star's cancellation ratio, written by the evaluations that accumulated
// A_TS (plain ones and the first stage of a step) and read by the others.
struct FinBufs {
    const double* in;
    double *X, *Y, *H1, *H2;
    const double* m;
    double* acc;
    float* kr;
    double* xr;          // rare_rows' sums (mixed form)
    const double* hp;    // hard_part's, or null if the pair kernel has none
    const JRec64* j64;   // this evaluation's records
    JRec64* jnext;       // the next one's (another buffer: other rows may
                         // still read this evaluation's)
};

// One row of a cluster's stars: local stars first .. first + 63 of the nst to
// be done (of the cluster's nall: fewer in an i shard), BH at index off; row:
// this one's index among all rows.
struct Row {
    int off, nst, first, row, nall;
};

// The workgroup's rows of a cluster: row q.row by all FG waves (G = FG), or
// rows q.row .. q.row + FG - 1 by one wave each (G = 1; q.first: the first
// star of the workgroup's).  Accelerations, stage update and BH shares, and,
// inside a step (STAGE 1..3), the records and row sums of the driver's next
// evaluation on the state the stage update gives.  Every thread calls this.
//
// bh (G = FG): lane k < 3 of the last wave gets the BH's component k, which
// fin_close takes from there.
//
// Q = 4 (with G = FG): group `sub` of 16 stars of row q.row only.  At n = 1025
// a row's 16 chunks of partials are 131 KB, which one CU reads in 4 us of
// k_fin's 9.5 (MI355X, by its clock); its four quarters go to four CUs.
//
// G = FG is for few rows: one wave adding all S chunks of its stars leaves
// most of the chip idle (at n = 10241, S = 128 that took as long as the pair
// kernel).  With many rows the chip is full either way, and the star part
// behind the gather, which one wave runs, counts: G = 1 keeps all FG busy.
template <int MODE, int STAGE, int G, int Q>
__device__ __forceinline__ void fin_rows(const FinBufs& F, const RowBufs& R, const Row& q,
                                         const void* __restrict__ part, int S, size_t stride,
                                         size_t idx0, const double* __restrict__ gsp,
                                         const int* __restrict__ flist,
                                         const int* __restrict__ fn, double m0, const MixPrep& M,
                                         const Phys& P, StageIn& bh, int sub)
{
    constexpr bool TS = STAGE <= 1;
    constexpr int RS = RB / Q;                      // stars per wave of the star part
    const int lane = threadIdx.x & 63, cap = P.cap;
    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int mine = G == 1 ? wid : 0;              // this wave's row of the workgroup's
    const int lf = q.first + mine * RB + sub * RS;  // its first star
    const int li = lf + lane % RS;
    const bool ok = li < q.nst && lane < RS;
    const int lc = li < q.nst ? li : min(q.first, q.nst - 1);
    const int p = q.off + 1 + lc;
    const bool star = G == 1 ? lf < q.nst : wid == 0;   // this wave runs the star part
    int nf = 0, hslot = -1;      // the lane's star: hard_part's slot of it
    bool is_hard = false;
    // the BH-close and hard stars, if any
    __shared__ double hx[MODE == 1 ? (G == 1 ? FG : 1) : 1][HSLOT][MODE == 1 ? NACC + 1 : 1];
    auto rare = [&]() {
        if (MODE == 0) return;
        nf = *fn;
        unsigned long long any = 0ull;
#pragma unroll
        for (int r = 0; r < (G == 1 ? FG : 1); ++r)
            if (q.first + r * RB < q.nst) {
                const unsigned long long hm = R.hmask[q.row + r];
                unsigned long long rest = hm;
                if (F.hp) {
                    rest &= rest - 1;
                    rest &= rest - 1;
                }
                if (Q > 1) rest = (rest >> (sub * RS)) & 0xffffu;
                any |= rest;
                if (r != mine) continue;
                const int bit = sub * RS + lane % RS;
                is_hard = (hm >> bit) & 1;
                if (F.hp && is_hard) {
                    const int before = __popcll(hm & ((1ull << bit) - 1ull));
                    hslot = before < HSLOT ? before : -1;
                }
                // by a wave each of those that have no star part (G = 1: by
                // the row's)
                if (F.hp && hm)
                    for (int k = 0; k < HSLOT && k < __popcll(hm); ++k)
                        if (G == 1 || wid == 1 + k) {
                            const double t =
                                hard_sum(F.hp + ((size_t)(q.row + r) * HSLOT + k) * HCHUNK * (NACC + 1), S);
                            if (MODE == 1 && lane <= NACC) hx[G == 1 ? wid : 0][k][lane] = t;
                        }
            }
        if (nf > 0 || any)
            rare_rows(F.j64, F.in, cap, P.eps2, q.off, Q > 1 ? min(q.nst, lf + RS) : q.nst,
                      Q > 1 ? lf : q.first, G == 1 ? FG : 1, R.hmask + q.row, sub * RS,
                      Q > 1 ? 0xffffull : ~0ull, q.nall, F.hp ? HSLOT : 0, flist, nf, F.xr);
    };
    static_assert(HSLOT == 2, "two bits cleared above");
    // everything the star part reads, requested ahead of the partial sums
    StageIn st;
    double gs[NGS], mp = 0.0, D2 = 0.0, e = 0.0, x0[3], x0n[3];
    float kr = 0.0f;
    double A[NACC + 1];
    if (G == 1) {
        rare();
        if (star) {
            D2 = F.j64[p].D2;
            e = F.j64[p].e;
            st = stage_load<STAGE>(F.in, F.X, F.H1, F.H2, cap, p);
            const StageIn b0 = stage_load<STAGE>(F.in, F.X, F.H1, F.H2, cap, q.off);
            mp = F.m[p];
#pragma unroll
            for (int k = 0; k < NGS; ++k) gs[k] = gsp[k];
            if (MODE == 1 && !TS) kr = F.kr[p];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                x0[k] = b0.x[k];
                x0n[k] = stage_pos<STAGE>(b0, P.dt, k);
            }
            gather_row<MODE, TS, G>(part, S, stride, idx0 + lc, M.mmax, A);
        }
    } else {
        // Row r of what the star part reads of its star: components of in, X,
        // H1 and H2 as the stage needs them, the mass, D2 and e.  Wave w
        // fetches rows w, w + FG, ... beside its partial sums, the last wave
        // also the BH's state and the separable sums (by lane: as scalar loads
        // they would queue, one line each, behind one another), all through
        // LDS; one trip to memory in all.
        constexpr int NST = STAGE == 3 ? 24 : STAGE == 2 ? 12 : 6, NR = NST + 3;
        constexpr int H = FG * Q, NL = (NR + H - 1) / H;
        const int h = wid * Q + (Q == 1 ? 0 : lane / RS);
        __shared__ double pre[NR][RS], uni[6 + NGS];
        double ld[NL], g0 = 0.0;
#pragma unroll
        for (int t = 0; t < NL; ++t) {
            const int r = h + t * H;
            ld[t] = 0.0;
            if (r < NST) {
                const double* b = r < 6 ? F.in : r < 12 ? F.X : r < 18 ? F.H1 : F.H2;
                ld[t] = b[(size_t)(r % 6) * cap + p];
            } else if (r < NR) {
                const double* b = r == NST ? F.m + p
                                           : r == NST + 1 ? &F.j64[p].D2 : &F.j64[p].e;
                ld[t] = *b;
            }
        }
        if (MODE == 1 && !TS && wid == 0) kr = F.kr[p];
        if (wid == FG - 1) {
            if (lane < 3) bh = stage_load<STAGE>(F.in, F.X, F.H1, F.H2, cap, q.off, lane, 1);
            if (lane < NGS) g0 = gsp[lane];
        }
        rare();
        if (Q == 1)
            gather_row<MODE, TS, G>(part, S, stride, idx0 + lc, M.mmax, A);
        else
            gather_sub<MODE, TS>(part, S, stride, idx0 + lc, M.mmax, A);
        const int ls = Q == 1 ? lane : lane % RS;
#pragma unroll
        for (int t = 0; t < NL; ++t)
            if (h + t * H < NR) pre[h + t * H][ls] = ld[t];
        if (wid == FG - 1) {
            if (lane < 3) {
                uni[lane] = bh.x[0];
                uni[3 + lane] = stage_pos<STAGE>(bh, P.dt, 0);
            }
            if (lane < NGS) uni[6 + lane] = g0;
        }
        __syncthreads();
        if (star) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                st.x[k] = pre[k][ls];
                st.v[k] = pre[3 + k][ls];
                if (STAGE >= 2) {
                    st.X[k] = pre[STAGE >= 2 ? 6 + k : 0][ls];
                    st.V[k] = pre[STAGE >= 2 ? 9 + k : 0][ls];
                }
                if (STAGE == 3) {
                    st.hx[k] = pre[STAGE == 3 ? 12 + k : 0][ls] + pre[STAGE == 3 ? 18 + k : 0][ls];
                    st.hv[k] = pre[STAGE == 3 ? 15 + k : 0][ls] + pre[STAGE == 3 ? 21 + k : 0][ls];
                }
                x0[k] = to_scalar(uni[k]);
                x0n[k] = to_scalar(uni[3 + k]);
            }
            mp = pre[NST][ls];
            D2 = pre[NST + 1][ls];
            e = pre[NST + 2][ls];
#pragma unroll
            for (int k = 0; k < NGS; ++k) gs[k] = to_scalar(uni[6 + k]);
        }
    }
    if (MODE == 1 && star && ok && (is_hard || nf > 0)) {
        // a hard star: its FP64 row instead of the gathered sums; another
        // one: plus its pairs with the BH-close stars
#pragma unroll
        for (int k = 0; k <= NACC; ++k)
            A[k] = hslot >= 0 ? hx[G == 1 ? wid : 0][hslot & (HSLOT - 1)][k]
                              : (is_hard ? 0.0 : A[k]) + F.xr[(size_t)k * cap + p];
    }
    if (!star) return;
    double cb[3] = {0.0, 0.0, 0.0}, a[3], nx[3], nv[3], g[NGS];
    bool f = false, hard = false;
    if (ok) {
        fin_star<STAGE>(st, x0, mp, D2, e, F.X, F.Y, F.H1, F.H2, cap, p, A, gs,
                        fin_consts(P, m0), F.acc, cb, a, nx, nv);
        if (MODE == 1 && TS) {
            kr = cancel_ratio(A[NACC], a);
            F.kr[p] = kr;
        }
        if (STAGE > 0) {
            f = prep_star(nx, nv, x0n, mp, p, m0, P.eps2, F.jnext, g, M, true, a, kr, hard);
        }
    }
    put_row<true, (STAGE > 0), Q>(q.row + mine, sub, ok, cb, g, R.rows, MODE == 1, f, hard, R.fmask,
                               R.hnext);
}

// A cluster without stars: its one row of zeros (all Q groups of it).
template <int Q>
__device__ __forceinline__ void empty_row(const RowBufs& R, int row, bool mixed)
{
    if (threadIdx.x < RV * Q) hand_over(&R.rows[(size_t)row * Q * RV + threadIdx.x], 0.0);
    if (mixed && threadIdx.x == 0) {
        hand_over(&R.fmask[row], 0ull);
        R.hnext[row] = 0ull;
    }
}

// After the last row of an evaluation: the BH at b0, its acceleration Newton
// sum_j m_j e_j^3 d_j plus lam times the rows' shares and its stage update
// (lane k of a wave: component k), and the next evaluation's separable sums and
// BH-close list.  PRE: the last wave holds the BH's state already (bh).
template <int MODE, int STAGE, bool PRE, int Q>
__device__ __forceinline__ void fin_close(const FinBufs& F, const RowBufs& R, int b0row,
                                          int b1row, int b0, double* __restrict__ gs,
                                          int* __restrict__ flist, int* __restrict__ fn,
                                          const Phys& P, const StageIn& bh)
{
    __shared__ double tot[RV];
    const int t = (int)threadIdx.x - (PRE ? (FG - 1) * 64 : 0);
    StageIn st = bh;
    double nwt = 0.0;
    if (t >= 0 && t < 3) {
        if (!PRE) st = stage_load<STAGE>(F.in, F.X, F.H1, F.H2, P.cap, b0, t, 1);
        nwt = gs[G_M1X + t];
    }
    rows_total<Q>(R.rows, b0row, b1row, tot);
    if (t >= 0 && t < 3) {
        double nx, nv;
        const double a = nwt + P.lam * tot[t];
        F.acc[(size_t)t * P.cap + b0] = a;
        stage_update<STAGE>(b0, P.cap, st, 0, t, a, F.X, F.Y, F.H1, F.H2, P.dt, nx, nv);
    }
    if (STAGE > 0) {
        __syncthreads();                       // gs has been read
        if (threadIdx.x < NGS) gs[threadIdx.x] = tot[RV_G + threadIdx.x];
        if (MODE == 1) list_flagged(R.fmask, b0row, b1row, b0 + 1, flist, fn);
    }
}

// Rows from row0 on, up to star p1 (all: the BH too, by the last workgroup;
// a sub-range is one i shard of a plain evaluation); the BH mass is m[0].  A
// workgroup per row and group of it (G = FG) or per FG rows (G = 1).
template <int MODE, int STAGE, int G, int Q>
__global__ __launch_bounds__(FWG) __attribute__((amdgpu_waves_per_eu(4, 8)))
void k_fin(FinBufs F, RowBufs R, const void* __restrict__ part, int S, MixPrep M, Phys P,
           int row0, int p1, int nrow)
{
    const int row = row0 + (G == 1 ? (int)blockIdx.x * FG : (int)blockIdx.x / Q);
    const Row q = {0, p1 - 1, row * RB, row, P.n - 1};
    StageIn bh = {};
    if (P.n > 1)
        fin_rows<MODE, STAGE, G, Q>(F, R, q, part, S, (size_t)P.cap, 1, R.gs, R.flist, R.fn,
                                    F.m[0], M, P, bh, (int)blockIdx.x % Q);
    else
        empty_row<Q>(R, 0, MODE == 1);
    if (R.ticket && last_block(R.ticket, gridDim.x)) {
        if (G > 1 && P.n > 1)
            fin_close<MODE, STAGE, true, Q>(F, R, 0, nrow, 0, R.gs, R.flist, R.fn, P, bh);
        else
            fin_close<MODE, STAGE, false, Q>(F, R, 0, nrow, 0, R.gs, R.flist, R.fn, P, bh);
    }
}

// k_fin of pn1_force_noalloc (FP64, G = FG): every workgroup adds the separable
// sums from k_prep's rows (prows, FWG threads: the order of k_prep's last
// workgroup) for itself, so that only one counter, R.ticket, is left, which
// k_prep clears in the same call.
template <int Q>
__global__ __launch_bounds__(FWG) __attribute__((amdgpu_waves_per_eu(4, 8)))
void k_fin_na(FinBufs F, RowBufs R, const double* __restrict__ prows,
              const void* __restrict__ part, int S, Phys P, int nrow)
{
    __shared__ double tot[RV];
    rows_total<Q>(prows, 0, nrow, tot);
    const int row = (int)blockIdx.x / Q;
    const Row q = {0, P.n - 1, row * RB, row, P.n - 1};
    StageIn bh = {};
    if (P.n > 1)
        fin_rows<0, 0, FG, Q>(F, R, q, part, S, (size_t)P.cap, 1, tot + RV_G, nullptr, nullptr,
                              F.m[0], MixPrep{}, P, bh, (int)blockIdx.x % Q);
    else
        empty_row<Q>(R, 0, false);
    if (last_block(R.ticket, gridDim.x))
        fin_close<0, 0, false, Q>(F, R, 0, nrow, 0, tot + RV_G, nullptr, nullptr, P, bh);
}

// ---------------------------------------------------------------------
// energy (FP64 in both modes)
// ---------------------------------------------------------------------
// The energy needs totals only (Limit-sticky9.c:452-550), so each unordered
// pair is evaluated once:
//   pot  -= m_i m_j w
//   pn2  += m_i m_j [w (Ae_i + Ae_j - 3.5 v_i.v_j) - 0.5 w^3 (r.v_i)(r.v_j)]
// with Ae = 1.5 |v|^2 + m0 e from the records.  Row a of 64 stars (one per
// lane) meets the stars of the next half of the rows, cyclically: rows a + 1
// .. a + h, h = nrow / 2 (a row less for the upper half of the rows when nrow
// is even), and its own stars above each lane's.  That list is split in S
// chunks of PW waves, which work as k_pair64w's.  Against all ordered pairs
// with five sums per star it is half the rsqrts and no partials: n = 65537,
// 4.17 -> 2.24 ms on MI355X (31 issue slots per pair: 2.17 ms at the FP64
// rate of 3.1e13 lanes/s).
// Chunks per row: 16, fewer while a wave's part would hold fewer than 4
// records (each meets half of the stars).
__host__ __device__ inline int energy_chunks(int nst)
{
    int s = 16;
    while (s > 1 && nst < 8 * s * PW) s >>= 1;
    return s;
}
constexpr int ECHUNK = 16;

// Per-lane constants of star i: position, p = -3.5 / sqrt(3/2) v, q = -0.5 /
// sqrt(3/2) v (the records hold s = sqrt(3/2) v).
struct IE64 {
    double x, y, z, px, py, pz, qx, qy, qz;
};

// One pair: a += m_j w, b += m_j [w (Ae_j - 3.5 v_i.v_j) - 0.5 w^3 (r.v_i)(r.v_j)].
__device__ __forceinline__ void ebody64(const JRec64& J, double mj, const IE64& I, double& a,
                                        double& b, double eps2)
{
    const double rx = J.x - I.x, ry = J.y - I.y, rz = J.z - I.z;
    const double R2e = __builtin_fma(rx, rx, __builtin_fma(ry, ry, __builtin_fma(rz, rz, eps2)));
    const double w = rsq64(R2e);
    const double rvi = __builtin_fma(I.qx, rx, __builtin_fma(I.qy, ry, I.qz * rz));
    const double rvj = __builtin_fma(J.sx, rx, __builtin_fma(J.sy, ry, J.sz * rz));
    double t = __builtin_fma(I.px, J.sx, __builtin_fma(I.py, J.sy, __builtin_fma(I.pz, J.sz, J.Ae)));
    t = __builtin_fma(w * w, rvi * rvj, t);
    const double mw = mj * w;
    a += mw;
    b = __builtin_fma(mw, t, b);
}

// Row `row` (of nrow) of a cluster's stars off + 1 .. off + nst, chunk s of S:
// its four sums {m v^2, -m m w, the pot_pn terms, the pot_pn2 terms} in out
// (LDS); the sums over single stars with chunk 0.  m0: the BH's mass, G1 =
// sum m e.  Every thread of the workgroup (PW waves) calls it.
constexpr int EV = 4;
__device__ __forceinline__ void energy_row(const JRec64* __restrict__ jr,
                                           const double* __restrict__ st, int cap, int off,
                                           int nst, int nrow, int row, int s, int S, double m0,
                                           double G1, double eps2, double* out)
{
    __shared__ double sh[PW][EV];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int li = row * RB + lane, p1 = off + 1;
    const bool ok = li < nst;
    const int i = p1 + (ok ? li : row * RB);
    const JRec64 me = jr[i];
    const double v[3] = {st[3 * cap + i], st[4 * cap + i], st[5 * cap + i]};
    IE64 I;
    I.x = me.x; I.y = me.y; I.z = me.z;
    I.px = -3.5 * PN1_ISQ15 * v[0]; I.py = -3.5 * PN1_ISQ15 * v[1]; I.pz = -3.5 * PN1_ISQ15 * v[2];
    I.qx = -0.5 * PN1_ISQ15 * v[0]; I.qy = -0.5 * PN1_ISQ15 * v[1]; I.qz = -0.5 * PN1_ISQ15 * v[2];
    // the list: stars [first, first + len) modulo nst
    const int h = nrow / 2 - ((nrow & 1) == 0 && row >= nrow / 2 ? 1 : 0);
    const int first = row + 1 < nrow ? (row + 1) * RB : 0, last = row + h;      // row of the end
    const int len = h <= 0 ? 0
                    : last < nrow ? min(nst, (last + 1) * RB) - (row + 1) * RB
                                  : max(nst - (row + 1) * RB, 0) + min(nst, (last - nrow + 1) * RB);
    const int part = (len + S * PW - 1) / (S * PW);
    const int q0 = min(len, (s * PW + wave) * part), q1 = min(len, q0 + part);
    double a = 0.0, b = 0.0;
    for (int j = first + q0; j < min(nst, first + q1); ++j) {
        const JRec64& J = jr[p1 + j];
        ebody64(J, J.m, I, a, b, eps2);
    }
    for (int j = max(first + q0 - nst, 0); j < first + q1 - nst; ++j) {
        const JRec64& J = jr[p1 + j];
        ebody64(J, J.m, I, a, b, eps2);
    }
    double t[EV] = {0.0, 0.0, 0.0, 0.0};
    if (s == 0) {
        // the row's own pairs, wave w taking records w, w + PW, ...
        for (int j = row * RB + wave; j < min(nst, row * RB + RB); j += PW) {
            const JRec64& J = jr[p1 + j];
            ebody64(J, j > li ? J.m : 0.0, I, a, b, eps2);
        }
        if (wave == 0) {
            // single-star terms of Limit-sticky9.c:452-550
            const double e = me.e, mp = me.m;
            double d[3], v0[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                d[k] = st[(size_t)k * cap + i] - st[(size_t)k * cap + off];
                v0[k] = st[(size_t)(3 + k) * cap + off];
            }
            const double V2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
            const double v0v = v0[0] * v[0] + v0[1] * v[1] + v0[2] * v[2];
            const double dv0 = d[0] * v0[0] + d[1] * v0[1] + d[2] * v0[2];
            const double dv = d[0] * v[0] + d[1] * v[1] + d[2] * v[2];
            t[0] = mp * V2;
            t[2] = 0.375 * mp * V2 * V2 + 1.5 * m0 * e * mp * V2 + 0.5 * m0 * m0 * e * e * mp
                   + 0.5 * m0 * e * mp * (3.0 * V2 - 7.0 * v0v - dv0 * dv * e * e);
            t[3] = mp * (0.5 * m0 * e * (G1 - mp * e));
        }
    }
    t[1] = -me.m * a;
    t[3] += me.m * __builtin_fma(me.Ae, a, b);
#pragma unroll
    for (int k = 0; k < EV; ++k) {
        const double u = wave_sum(ok ? t[k] : 0.0);
        if (lane == 0) sh[wave][k] = u;
    }
    __syncthreads();
    if (threadIdx.x < EV) {
        double u = sh[0][threadIdx.x];
#pragma unroll
        for (int w = 1; w < PW; ++w) u += sh[w][threadIdx.x];
        out[threadIdx.x] = u;
    }
    __syncthreads();
}

// The energy {kin, pot, pot_pn / c^2, pot_pn2 / c^2, total} of the cluster
// with its BH at off from the sums of its `cnt` workgroups (EV values each, S
// per row, rows `stride` workgroups apart), by a workgroup of PW waves.
__device__ __forceinline__ void energy_total(const double* eb, int cnt, int S, int stride,
                                             const double* __restrict__ st, int cap, int off,
                                             double m0, double G1, double lam,
                                             double* __restrict__ out)
{
    __shared__ double sh[PW][EV], tot[EV];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double t = 0.0;
#pragma unroll 8
    for (int k = (int)threadIdx.x / EV; k < cnt; k += PW * RB / EV)
        t += take_over(&eb[((size_t)(k / S) * stride + k % S) * EV + (threadIdx.x & (EV - 1))]);
#pragma unroll
    for (int off2 = EV; off2 < 64; off2 <<= 1) t += __shfl_xor(t, off2, 64);
    if (lane < EV) sh[wave][lane] = t;
    __syncthreads();
    if (threadIdx.x < EV) {
        t = sh[0][threadIdx.x];
#pragma unroll
        for (int w = 1; w < PW; ++w) t += sh[w][threadIdx.x];
        tot[threadIdx.x] = t;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const double v0x = st[3 * cap + off], v0y = st[4 * cap + off], v0z = st[5 * cap + off];
        const double kin = 0.5 * (m0 * (v0x * v0x + v0y * v0y + v0z * v0z) + tot[0]);
        const double pot = tot[1] - m0 * G1;
        const double pn = lam * tot[2], pn2 = lam * tot[3];
        out[0] = kin;
        out[1] = pot;
        out[2] = pn;
        out[3] = pn2;
        out[4] = kin + pot + pn + pn2;
    }
}

// Row and chunk of this workgroup of a grid of (rows, chunks): consecutive
// workgroups take the chunks of one row, so that an XCD's share of the
// resident ones reads two of a row's chunks and not all records (n = 65537:
// 2.24 ms, 2.44 with consecutive rows).  The grid is two-dimensional because a
// dimension holds less than 2^32 threads.
__device__ __forceinline__ int2 energy_item()
{
    const unsigned k = blockIdx.y * gridDim.x + blockIdx.x;
    return make_int2((int)(k / gridDim.y), (int)(k % gridDim.y));
}

// One workgroup per (row, chunk), the last one adds them up.  The
// BH mass is m0, the separable sums gs as k_prep left them.
inline __global__ __launch_bounds__(PW * RB)
void k_energy(const JRec64* __restrict__ jr, const double* __restrict__ st,
              const double* __restrict__ gs, double* __restrict__ eb, double* __restrict__ out,
              unsigned int* __restrict__ ticket, Phys P)
{
    __shared__ double t[EV];
    const int nrow = (int)gridDim.x, S = (int)gridDim.y;
    const int2 w = energy_item();
    const double G1 = gs[G_G1];
    if (P.n > 1)
        energy_row(jr, st, P.cap, 0, P.n - 1, nrow, w.x, w.y, S, P.m0, G1, P.eps2, t);
    else if (threadIdx.x < EV)
        t[threadIdx.x] = 0.0;
    if (threadIdx.x < EV)
        hand_over(&eb[((size_t)w.x * S + w.y) * EV + threadIdx.x], t[threadIdx.x]);
    if (last_block(ticket, (unsigned)(nrow * S)))
        energy_total(eb, nrow * S, S, S, st, P.cap, 0, P.m0, G1, P.lam, out);
}

}  // namespace pn1dev
