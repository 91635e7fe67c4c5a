// pn1_adj_rev.hpp -- one reverse sweep of the pair term phi_ij that gives
// the i-side and the j-side gradient together (the single-pass force VJP).
//
// phi_ij (adj_pair_phi, Limit-sticky9.c:39-51, 118-174, 278-382) carries a
// factor m_j in every term: phi = m_j psi with
//   psi = w3 G + lam H,  w = (|r|^2 + eps^2)^-1/2, w2 = w^2, w3 = w^3,
//   G = (u_i.r) E + lam b6 (u_i.dv) - Kh (u_0.r),
//       E = 1 + lam (m0 bb2 + b5)
//   H = -Ka bb1 + Kb e_j^3 (w - e_i)(u_i.d_j) + Kf br
//       + Kc (v_i.v_j) + Kd (v_j.d_i) + Ke (u_i.v_j) + Kg (u_0.v_j)
// with r = x_j - x_i, dv = v_j - v_i, t = |d_i|^2 - |r|^2,
//   b5 = |v_i|^2 - 2|dv|^2 + 1.5 (v_j.r)^2 w2,  b6 = 4 v_i.r - 3 v_j.r,
//   bb1 = 4w + 1.25 e_j + 0.25 t e_j^3,  bb2 = 4 e_i + 1.25 e_j - 0.25 t e_j^3,
//   br = 4 e_j + 1.25 w + 0.25 (|d_i|^2 - |d_j|^2) w3,
// and the i-only coefficients (m_i, e_i, d_i, v_i, u_i; m0, 1/m0, u_0)
//   Ka = m0 e_i^3 (u_i.d_i)            Kb = 3.5 m0
//   Kc = 4 e_i^3 (u_i.d_i - m_i/m0 u_0.d_i)
//   Kd = -3 e_i^3 (u_i.v_i) + 4 m_i e_i^3/m0 (u_0.v_i)
//   Ke = -4 e_i^3 (v_i.d_i)            Kf = m_i e_i^3 (u_0.d_i)
//   Kg = 3 m_i e_i^3/m0 (v_i.d_i)      Kh = 3.5 lam m_i e_i.
// This is adj_pair_phi regrouped (the same terms, summed in another order).
//
// The last four terms of H are products of an i-only and a j-only factor:
// their sums over j (or i) need only sum m_j v_j and sums of the K's over the
// stars, so they are no work of the pair loop (rev_sep states them per pair;
// k_adj_fin adds them from those sums, less the star's own share).  rev_core
// differentiates the rest by hand in reverse order.  Its gradient splits
// three ways:
//   * pair-level occurrences of x_i, v_i, x_j, v_j (through r, dv and the
//     dot products) go into per-pair vector accumulators;
//   * the i-only scalars (e_i^3, u_i.d_i, ..., |d_i|^2, m0) enter psi
//     through the K's, E, bb2, t and Kh: their adjoints are linear in a
//     handful of pair sums (SA ... RB2), accumulated per pair and chained to
//     (x_i, v_i, m0) once per lane by rev_ifin;
//   * the j-only scalars |d_j|^2, e_j, e_j^3 and |v_j|^2 need two sums, A2
//     and R1, which rev_jfin chains to (x_j, v_j).
// Everything of one star that the sweep multiplies by (RevD) is formed once
// per star, not per pair.  Positions enter only through differences, so with
// d = x - x_BH the BH position gradient is minus the stars' sum (handled by
// the caller); the pair term does not depend on the BH velocity.
#pragma once
#include "pn1_adj_kernels.hpp"
#include "pn1_rows.hpp"

namespace pn1dev {

// Lane constants of star i (read-only in the j loop): w4 = 4 lam v,
// rb2e = |d|^2 + eps^2, Ei = 1 + lam (4 m0 e - |v|^2), T = |d|^2 / 4, nKa =
// -lam Ka, Kfl = lam Kf; the K's of the separable terms.
struct RevI {
    double x[3], v[3], d[3], u[3], w4[3];
    double rb2e, rbe, uivi, Ei, T, nKa, Kfl, Kh;
    double Kc, Kd, Ke, Kg;
};

// Per-lane sums over j of the i side; mv = sum m_j v_j and qs = sum of RevD's
// Qd belong to the separable terms.
struct RevIAcc {
    double gx[3], br3[3], gv3[3];
    double SA, Sq, SF, SH, SM, SR, SW, RB2;
    double mv[3], qs[3];
};

// Star j as a record, and its sums over i; t, ka, kf, kg = m_j times the sums
// of lam (Kc v_i + Kd d_i + Ke u_i), -lam Ka, lam Kf and lam Kg belong to the
// separable terms.
struct RevJ {
    double x[3], v[3], rc2, rce, m;
};
struct RevJAcc {
    double gx[3], gv[3], A2, R1;
    double t[3], ka, kf, kg;
};

// What the sweep needs of star j, with its weight P (m_j, or 0 for no pair):
//   E2 = -2 lam |v|^2          Y = 1.25 lam m0 e     B = 0.25 lam m0 e^3
//   D = 1.25 e, C = 0.25 e^3   e4 = 4 e              T = |d|^2 / 4
//   c = 3.5 lam m0 P e^3, Qd = c d                   h = (|d|^2 + eps^2) / 6
constexpr int REVD_F = 19;
struct RevD {
    double x[3], v[3], P, E2, Y, B, D, C, e4, T, c, Qd[3], h;
};

// Uniform values of one evaluation.
struct RevU {
    double x0[3], u0[3], m0, im0, Kb, eps2, lam;
};

__host__ __device__ __forceinline__ RevU rev_uniform(const ABH& B, double eps2, double lam)
{
    RevU U;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        U.x0[k] = B.x0[k];
        U.u0[k] = B.u0[k];
    }
    U.m0 = B.m0;
    U.im0 = 1.0 / B.m0;
    U.Kb = 3.5 * B.m0;
    U.eps2 = eps2;
    U.lam = lam;
    return U;
}

__host__ __device__ __forceinline__ RevI rev_setup(const ARec& me, const RevU& U)
{
    RevI I;
    I.x[0] = me.x; I.x[1] = me.y; I.x[2] = me.z;
    I.v[0] = me.vx; I.v[1] = me.vy; I.v[2] = me.vz;
    I.d[0] = me.dx; I.d[1] = me.dy; I.d[2] = me.dz;
    I.u[0] = me.ux; I.u[1] = me.uy; I.u[2] = me.uz;
#pragma unroll
    for (int k = 0; k < 3; ++k) I.w4[k] = 4.0 * U.lam * I.v[k];
    I.rb2e = me.D2 + U.eps2;
    I.rbe = me.e;
    I.T = 0.25 * me.D2;
    const double rbe3 = me.e * me.e * me.e;
    const double uidi = dot(I.u, I.d), u0di = dot(U.u0, I.d);
    const double u0vi = dot(U.u0, I.v), vidi = dot(I.v, I.d);
    I.uivi = dot(I.u, I.v);
    I.Ei = 1.0 + U.lam * (4.0 * U.m0 * me.e - dot(I.v, I.v));
    const double mi = me.m, mim0 = mi * U.im0;
    I.nKa = -U.lam * U.m0 * rbe3 * uidi;
    I.Kc = 4.0 * rbe3 * (uidi - mim0 * u0di);
    I.Kd = rbe3 * (-3.0 * I.uivi + 4.0 * mim0 * u0vi);
    I.Ke = -4.0 * rbe3 * vidi;
    I.Kfl = U.lam * mi * rbe3 * u0di;
    I.Kg = 3.0 * mim0 * rbe3 * vidi;
    I.Kh = 3.5 * U.lam * mi * me.e;
    return I;
}

__host__ __device__ __forceinline__ RevJ rev_jrec(const ARec& r)
{
    RevJ J;
    J.x[0] = r.x; J.x[1] = r.y; J.x[2] = r.z;
    J.v[0] = r.vx; J.v[1] = r.vy; J.v[2] = r.vz;
    J.rc2 = r.D2;
    J.rce = r.e;
    J.m = r.m;
    return J;
}

__host__ __device__ __forceinline__ RevD rev_derive(const RevJ& J, const RevU& U, double P)
{
    RevD R;
    const double e = J.rce, e3 = e * e * e, lm0 = U.lam * U.m0;
    R.P = P;
    R.c = U.lam * U.Kb * P * e3;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        R.x[k] = J.x[k];
        R.v[k] = J.v[k];
        R.Qd[k] = R.c * (J.x[k] - U.x0[k]);
    }
    R.E2 = -2.0 * U.lam * dot(J.v, J.v);
    R.D = 1.25 * e;
    R.C = 0.25 * e3;
    R.Y = lm0 * R.D;
    R.B = lm0 * R.C;
    R.e4 = 4.0 * e;
    R.T = 0.25 * J.rc2;
    R.h = (J.rc2 + U.eps2) / 6.0;
    return R;
}

__host__ __device__ __forceinline__ void rev_zero(RevIAcc& a)
{
#pragma unroll
    for (int k = 0; k < 3; ++k) a.gx[k] = a.br3[k] = a.gv3[k] = a.mv[k] = a.qs[k] = 0.0;
    a.SA = a.Sq = a.SF = a.SH = a.SM = a.SR = a.SW = a.RB2 = 0.0;
}

__host__ __device__ __forceinline__ void rev_zero(RevJAcc& a)
{
#pragma unroll
    for (int k = 0; k < 3; ++k) a.gx[k] = a.gv[k] = a.t[k] = 0.0;
    a.A2 = a.R1 = a.ka = a.kf = a.kg = 0.0;
}

// One pair (i, j): adds P d (psi less its separable terms) / d(...) to both
// sides' pair sums.
__host__ __device__ __forceinline__ void rev_core(const RevI& I, const RevD& J, const RevU& U,
                                                  RevIAcc& ai, RevJAcc& aj)
{
    // every product goes into an FMA where one follows (fma: the host build
    // of the check, too)
    const auto fma = [](double a, double b, double c) { return __builtin_fma(a, b, c); };
    const double P = J.P, lam3 = 3.0 * U.lam, lam15 = 1.5 * U.lam, lm0 = U.lam * U.m0;
    // ---- forward ----
    double r[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) r[k] = J.x[k] - I.x[k];
    const double R2e = fma(r[0], r[0], fma(r[1], r[1], fma(r[2], r[2], U.eps2)));
    const double w = rsq64(R2e);
    const double w2 = w * w, w3 = w2 * w;
    const double t = I.rb2e - R2e;
    const double vjr = fma(J.v[0], r[0], fma(J.v[1], r[1], J.v[2] * r[2]));
    const double tv = vjr * w, tl = lam15 * tv;
    const double y = fma(-J.B, t, J.Y);                      // lam m0 (bb2 - 4 e_i)
    double E = fma(I.w4[0], J.v[0], fma(I.w4[1], J.v[1], fma(I.w4[2], J.v[2], I.Ei + J.E2)));
    E = fma(tl, tv, E) + y;
    const double b6 = fma(-lam3, vjr, fma(I.w4[0], r[0], fma(I.w4[1], r[1], I.w4[2] * r[2])));
    const double uir = fma(I.u[0], r[0], fma(I.u[1], r[1], I.u[2] * r[2]));
    const double u0r = fma(U.u0[0], r[0], fma(U.u0[1], r[1], U.u0[2] * r[2]));
    const double uiw = fma(I.u[0], J.v[0], fma(I.u[1], J.v[1], fma(I.u[2], J.v[2], -I.uivi)));
    const double qd = fma(I.u[0], J.Qd[0], fma(I.u[1], J.Qd[1], I.u[2] * J.Qd[2]));
    const double bb1 = fma(4.0, w, fma(J.C, t, J.D));
    const double tb = I.T - J.T;
    const double br = fma(tb, w3, fma(1.25, w, J.e4));
    const double G = fma(uir, E, fma(b6, uiw, -(I.Kh * u0r)));
    // ---- reverse: P (w3 G + nKa bb1 + Kfl br) + (w - e_i) qd ----
    const double g3 = P * w3;
    const double gE = g3 * E, gur = g3 * uir, b6b = g3 * uiw, uiwb = g3 * b6;
    const double u0rb = -(g3 * I.Kh);
    const double g2 = tl * gur, g2d = g2 + g2;
    const double vjrb = fma(g2d, w, -(lam3 * b6b));
    const double bb1b = P * I.nKa;
    const double x2 = fma(-lm0, gur, bb1b), tbar = J.C * x2;
    const double brb = P * I.Kfl, tbb = w3 * brb;
    const double w3b = fma(tb, brb, P * G);
    const double wme = w - I.rbe;
    const double qw = qd * wme, cw = J.c * wme;
    double wb = fma(4.0, bb1b, qd);
    wb = fma(1.25, brb, wb);
    wb = fma(g2d, vjr, wb);
    wb = fma(3.0 * w2, w3b, wb);
    const double al = fma(-2.0, tbar, -(w3 * wb));
    // ---- sums ----
    ai.SA = fma(P, bb1, ai.SA);
    ai.Sq += qw;
    ai.SF = fma(P, br, ai.SF);
    ai.SH = fma(g3, u0r, ai.SH);
    ai.SM = fma(gur, y, ai.SM);
    ai.SR += gur;
    ai.SW += uiwb;
    ai.RB2 = fma(0.25, tbb, ai.RB2 + tbar);
    aj.A2 += gur;
    aj.R1 = fma(t, tbar, fma(J.h, tbb, aj.R1 + qw));
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double rb = fma(al, r[k], fma(vjrb, J.v[k], fma(b6b, I.w4[k],
                                                            fma(gE, I.u[k], u0rb * U.u0[k]))));
        ai.gx[k] -= rb;
        aj.gx[k] = fma(cw, I.u[k], aj.gx[k] + rb);
        ai.br3[k] = fma(b6b, r[k], ai.br3[k]);
        ai.gv3[k] = fma(gur, J.v[k], ai.gv3[k]);
        aj.gv[k] = fma(vjrb, r[k], fma(gur, I.w4[k], fma(uiwb, I.u[k], aj.gv[k])));
    }
}

// The separable terms of one pair.
__host__ __device__ __forceinline__ void rev_sep(const RevI& I, const RevD& J, const RevU& U,
                                                 RevIAcc& ai, RevJAcc& aj)
{
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        ai.mv[k] += J.P * J.v[k];
        ai.qs[k] += J.Qd[k];
        aj.t[k] += J.P * U.lam * (I.Kc * I.v[k] + I.Kd * I.d[k] + I.Ke * I.u[k]);
    }
    aj.ka += J.P * I.nKa;
    aj.kf += J.P * I.Kfl;
    aj.kg += J.P * U.lam * I.Kg;
}

// One pair (i, j) with weight P, all terms.
__host__ __device__ __forceinline__ void rev_pair(const RevI& I, const RevJ& J, const RevU& U,
                                                  double P, RevIAcc& ai, RevJAcc& aj)
{
    const RevD D = rev_derive(J, U, P);
    rev_core(I, D, U, ai, aj);
    rev_sep(I, D, U, ai, aj);
}

// i side of the lane's star: g = d/d(x_i, v_i, m0) of the pair sums,
// from the accumulators and the record `me`.
__host__ __device__ __forceinline__ void rev_ifin(const ARec& me, const RevU& U,
                                                  const RevIAcc& a, double (&g)[NADJ1])
{
    const double lam = U.lam, m0 = U.m0, im0 = U.im0, mi = me.m;
    const double vi[3] = {me.vx, me.vy, me.vz}, di[3] = {me.dx, me.dy, me.dz};
    const double ui[3] = {me.ux, me.uy, me.uz};
    const double rbe = me.e, rbe2 = rbe * rbe, rbe3 = rbe2 * rbe;
    const double uidi = dot(ui, di), u0di = dot(U.u0, di), u0vi = dot(U.u0, vi);
    const double vidi = dot(vi, di), uivi = dot(ui, vi);
    const double mim0 = mi * im0;
    // adjoints of the K's (Kb: its share of the m0 derivative is Sq / m0)
    const double Kab = -lam * a.SA, Kcb = lam * dot(vi, a.mv), Kdb = lam * dot(di, a.mv);
    const double Keb = lam * dot(ui, a.mv), Kfb = lam * a.SF, Kgb = lam * dot(U.u0, a.mv);
    const double Khb = -a.SH;
    // m0 directly (E, Ka, Kb) and through 1/m0 (Kc, Kd, Kg)
    double m0b = 4.0 * lam * rbe * a.SR + im0 * (a.SM + a.Sq) + Kab * rbe3 * uidi;
    const double im0b = mi * rbe3 * (-4.0 * Kcb * u0di + 4.0 * Kdb * u0vi + 3.0 * Kgb * vidi);
    m0b -= im0 * im0 * im0b;
    const double rbe3b = Kab * m0 * uidi + Kcb * 4.0 * (uidi - mim0 * u0di)
                         + Kdb * (-3.0 * uivi + 4.0 * mim0 * u0vi) - 4.0 * Keb * vidi
                         + Kfb * mi * u0di + 3.0 * Kgb * mim0 * vidi;
    const double uidib = Kab * m0 * rbe3 + 4.0 * Kcb * rbe3;
    const double u0dib = -4.0 * Kcb * rbe3 * mim0 + Kfb * mi * rbe3;
    const double uivib = -3.0 * Kdb * rbe3 - a.SW;
    const double u0vib = 4.0 * Kdb * mi * rbe3 * im0;
    const double vidib = -4.0 * Keb * rbe3 + 3.0 * Kgb * mim0 * rbe3;
    const double rbeb = 3.5 * lam * mi * Khb + 4.0 * lam * m0 * a.SR - dot(ui, a.qs)
                        + 3.0 * rbe2 * rbe3b;
    const double rb2b = a.RB2 - 0.5 * rbe3 * rbeb;
    // the separable terms' vectors: lam Kd sum m_j v_j and lam Kc sum m_j v_j
    const double Kc = lam * 4.0 * rbe3 * (uidi - mim0 * u0di);
    const double Kd = lam * rbe3 * (-3.0 * uivi + 4.0 * mim0 * u0vi);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double db = 2.0 * rb2b * di[k] + uidib * ui[k] + u0dib * U.u0[k] + vidib * vi[k];
        g[k] = a.gx[k] + Kd * a.mv[k] + db;
        g[3 + k] = 4.0 * lam * (a.br3[k] + a.gv3[k]) + Kc * a.mv[k] - 2.0 * lam * a.SR * vi[k]
                   + uivib * ui[k] + u0vib * U.u0[k] + vidib * di[k];
    }
    g[6] = m0b;
}

// j side of the record J: g = d/d(x_j, v_j) of the pair sums.
__host__ __device__ __forceinline__ void rev_jfin(const RevJ& J, const RevU& U, const RevJAcc& a,
                                                  double (&g)[NADJ2])
{
    const double e = J.rce, e2 = e * e, e3 = e2 * e;
    // adjoint of |d_j|^2, directly and through e_j and e_j^3
    const double rho = -1.5 * e2 * a.R1
                       - 0.5 * e3 * (1.25 * (U.lam * U.m0 * a.A2 + a.ka) + 4.0 * a.kf);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        g[k] = a.gx[k] + 2.0 * rho * (J.x[k] - U.x0[k]);
        g[3 + k] = a.gv[k] - 4.0 * U.lam * a.A2 * J.v[k] + a.t[k] + a.kg * U.u0[k];
    }
}


// =====================================================================
// Device: the single-pass pair kernel.
//
// A workgroup (4 waves) takes 256 stars i (one per lane, fixed) and a
// chunk of j records, in tiles of 64.  The tile's records (RevD, prepared
// once per star and evaluation) are staged in LDS, one copy for the four
// waves, read-only for the tile.  Step t pairs lane l with record
// jt + ((l + t) mod 64), read from LDS, while that record's running j-side
// sums move one lane down after every step (a DPP lane rotation).  So each
// lane meets every record of the tile once and, after 64 steps, every
// record's sums are back on its home lane, summed over the wave's 64 stars.
// The four waves' sums are added in wave order through LDS and written per
// (i block, j); the i side is written per (j chunk, i).  Every order is
// fixed, so the result is bitwise reproducible.
//
// Bound: FP64 issue.  151 VALU instructions per pair (129 FP64, 16 DPP
// moves) against 231 before the separable terms left the loop and the
// records' products were formed once per star: at n = 16385 on MI355X 1.32 ms
// per launch instead of 1.91 (2.0e11 pairs/s), 87% of what those
// instructions take at the card's FP64 rate.
// =====================================================================
// The value v of lane (lane + 1) mod 64: DPP wave_rol:1 on each half
// (v_mov_b32_dpp, a VALU move with no LDS round trip, so nothing waits on
// it; measured 12% faster for this kernel than ds_bpermute).  The records
// themselves are read from LDS instead (another 3%: their moves leave the
// VALU).
__device__ __forceinline__ double lane_next(double v)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)b, 0x134, 0xf, 0xf, true);
    const unsigned hi =
        (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), 0x134, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

__device__ __forceinline__ void rev_next(RevJAcc& a)
{
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        a.gx[k] = lane_next(a.gx[k]);
        a.gv[k] = lane_next(a.gv[k]);
    }
    a.A2 = lane_next(a.A2);
    a.R1 = lane_next(a.R1);
}

// RevD as REVD_F fields, in memory [REVD_F][cap] and, two fields to a 16-byte
// read, in the LDS tile [REVD_F2][64 + 1] (the lanes read records (l + t) mod
// 64, consecutive: no bank conflicts; slot 64 is an empty record).
constexpr int REV_SLOTS = 65;
constexpr int REVD_F2 = (REVD_F + 1) / 2;
constexpr int REV_JS = 8;                    // j-side sums that travel
__device__ __forceinline__ void revd_put(const RevD& R, double* __restrict__ jd, size_t cap,
                                         int p)
{
    const double f[REVD_F] = {R.x[0], R.x[1], R.x[2], R.v[0], R.v[1], R.v[2], R.P,
                              R.E2, R.Y, R.B, R.D, R.C, R.e4, R.T, R.c, R.Qd[0], R.Qd[1],
                              R.Qd[2], R.h};
#pragma unroll
    for (int k = 0; k < REVD_F; ++k) jd[k * cap + p] = f[k];
}
__device__ __forceinline__ RevD revd_get(const double2 (*tl)[REV_SLOTS], int slot)
{
    double f[2 * REVD_F2];
#pragma unroll
    for (int k = 0; k < REVD_F2; ++k) {
        const double2 d = tl[k][slot];
        f[2 * k] = d.x;
        f[2 * k + 1] = d.y;
    }
    RevD R;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        R.x[k] = f[k];
        R.v[k] = f[3 + k];
        R.Qd[k] = f[15 + k];
    }
    R.P = f[6]; R.E2 = f[7]; R.Y = f[8]; R.B = f[9]; R.D = f[10]; R.C = f[11];
    R.e4 = f[12]; R.T = f[13]; R.c = f[14]; R.h = f[18];
    return R;
}

// The workgroup's stars (lane: star i, weightless unless iok) against
// records [j0, j1): the i side's sums in g (d/d(x_i, v_i, m0)), the j side's
// given to putj(j, {d/d(x_j, v_j)}) by wave 0.  live (wave-uniform) is false
// for a wave past the last star of a partly filled i block: it skips the
// steps (it still stages and meets the barriers).  Every thread calls it.
template <class PutJ>
__device__ __forceinline__ void rev_chunk(const ARec* __restrict__ rec,
                                          const double* __restrict__ jd, size_t cap,
                                          const RevU& U, int i, bool iok, bool live, int j0,
                                          int j1, double (&g)[NADJ1], PutJ putj)
{
    __shared__ double2 tl[REVD_F2][REV_SLOTS];
    __shared__ double sh[REV_JS][WG / 64][64];
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = (int)(threadIdx.x & 63);
    ARec me = rec[i];
    if (!iok) me.ux = me.uy = me.uz = me.m = 0.0;     // every term is linear in (u_i, m_i)
    const RevI I = rev_setup(me, U);
    RevIAcc ai;
    rev_zero(ai);
    if (threadIdx.x < REVD_F2) tl[threadIdx.x][64] = make_double2(0.0, 0.0);
    for (int jt = j0; jt < j1; jt += 64) {
        const int jl = jt + lane;
#pragma unroll
        for (int f = wv; f < REVD_F; f += WG / 64)
            reinterpret_cast<double*>(&tl[f / 2][lane])[f & 1] = jl < j1 ? jd[f * cap + jl] : 0.0;
        __syncthreads();
        RevJAcc aj;
        rev_zero(aj);
        if (live) {
#pragma unroll 1
            for (int t = 0; t < 64; ++t) {
                const int slot = (lane + t) & 63;
                rev_core(I, revd_get(tl, jt + slot == i ? 64 : slot), U, ai, aj);
                rev_next(aj);
            }
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            sh[k][wv][lane] = aj.gx[k];
            sh[3 + k][wv][lane] = aj.gv[k];
        }
        sh[6][wv][lane] = aj.A2;
        sh[7][wv][lane] = aj.R1;
        __syncthreads();
        if (wv == 0 && jl < j1) {
            double s[REV_JS];
#pragma unroll
            for (int k = 0; k < REV_JS; ++k)
                s[k] = ((sh[k][0][lane] + sh[k][1][lane]) + sh[k][2][lane]) + sh[k][3][lane];
            RevJAcc t;
            rev_zero(t);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                t.gx[k] = s[k];
                t.gv[k] = s[3 + k];
            }
            t.A2 = s[6];
            t.R1 = s[7];
            double gj[NADJ2];
            rev_jfin(rev_jrec(rec[jl]), U, t, gj);
            putj(jl, gj);
        }
    }
    rev_ifin(me, U, ai, g);
}


// Block (s, ib): stars 1 + ib*WG + [0, WG), records [1 + s L, 1 + (s+1) L).
// part rows: i side (s*NADJ1 + k)*cap + i, s < S; j side
// (S*NADJ1 + ib*NADJ2 + k)*cap + j.
__global__ __launch_bounds__(WG) void k_adj_rev(const ARec* __restrict__ rec,
                                               const double* __restrict__ jd,
                                               const double* __restrict__ y,
                                               const double* __restrict__ mu,
                                               const double* __restrict__ m,
                                               double* __restrict__ part, Phys P, int L, int S)
{
    const int s = (int)blockIdx.x % S, ib = (int)blockIdx.x / S;
    const int n = P.n;
    const size_t cap = (size_t)P.cap;
    const int li = ib * WG + (int)threadIdx.x + 1;
    const bool iok = li < n;
    const bool live = ib * WG + (__builtin_amdgcn_readfirstlane((int)threadIdx.x) & ~63) + 1 < n;
    const int j0 = 1 + s * L, j1 = min(n, j0 + L);
    const RevU U = rev_uniform(load_abh(y, mu, m, P.cap, 0), P.eps2, P.lam);
    double* pj = part + ((size_t)S * NADJ1 + (size_t)ib * NADJ2) * cap;
    double g[NADJ1];
    rev_chunk(rec, jd, cap, U, iok ? li : n - 1, iok, live, j0, j1, g,
              [&](int j, const double (&gj)[NADJ2]) {
#pragma unroll
                  for (int k = 0; k < NADJ2; ++k) pj[(size_t)k * cap + j] = gj[k];
              });
    if (iok) {
#pragma unroll
        for (int k = 0; k < NADJ1; ++k) part[((size_t)s * NADJ1 + k) * cap + li] = g[k];
    }
}

// ---------------------------------------------------------------------
// The O(n) kernels of the VJP, on rows of 64 stars as the force's.
// ---------------------------------------------------------------------
// A row's values of k_adj_prep: the sums over all stars of
//   m v (0..2), Qd (3..5), lam (Kc v + Kd d + Ke u) (6..8), -lam Ka, lam Kf,
//   lam Kg (9, 10, 11)
// and of k_adj_fin: of its stars' g_x (0..2) and d/dm0 (3).
//
// The cotangent mu of one stage's VJP is a A + b B (B may be null).
struct AdjLin {
    const double *A, *B;
    double a, b;
};
__device__ __forceinline__ double adj_lin(const AdjLin& l, size_t i)
{
    double r = l.a * l.A[i];
    if (l.B) r += l.b * l.B[i];
    return r;
}

// Row of stars p (ok) of the cluster whose BH is at b0: mu, the records
// (ARec, RevD) and the row's sums.  Every lane of the wave calls it.
__device__ __forceinline__ void adj_prep_row(const double* __restrict__ y, const AdjLin& l,
                                             double* __restrict__ mu,
                                             const double* __restrict__ m, size_t cap,
                                             double eps2, double lam, int p, bool ok, int b0,
                                             ARec* __restrict__ rec, double* __restrict__ jd,
                                             double* __restrict__ rows, int row)
{
    const int lane = threadIdx.x & 63;
    double v[RV];
#pragma unroll
    for (int k = 0; k < RV; ++k) v[k] = 0.0;
    if (ok) {
        ABH B;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            B.x0[k] = y[k * cap + b0];
            B.u0[k] = adj_lin(l, (3 + k) * cap + b0);
        }
        B.m0 = m[b0];
        double u[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) mu[k * cap + p] = u[k] = adj_lin(l, k * cap + p);
        ARec r;
        r.x = y[p]; r.y = y[cap + p]; r.z = y[2 * cap + p];
        r.vx = y[3 * cap + p]; r.vy = y[4 * cap + p]; r.vz = y[5 * cap + p];
        r.ux = u[3]; r.uy = u[4]; r.uz = u[5];
        r.m = m[p];
        r.dx = r.x - B.x0[0]; r.dy = r.y - B.x0[1]; r.dz = r.z - B.x0[2];
        r.D2 = r.dx * r.dx + r.dy * r.dy + r.dz * r.dz;
        r.e = rsq64(r.D2 + eps2);
        r.pad = 0.0;
        rec[p] = r;
        const RevU U = rev_uniform(B, eps2, lam);
        const RevI I = rev_setup(r, U);
        const RevD D = rev_derive(rev_jrec(r), U, r.m);
        revd_put(D, jd, cap, p);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            v[k] = r.m * I.v[k];
            v[3 + k] = D.Qd[k];
            v[6 + k] = lam * (I.Kc * I.v[k] + I.Kd * I.d[k] + I.Ke * I.u[k]);
        }
        v[9] = I.nKa;
        v[10] = I.Kfl;
        v[11] = lam * I.Kg;
    }
    const double t = wave_sums16(v);
    if ((lane & 3) == 0) hand_over(&rows[(size_t)row * RV + (lane >> 2)], t);
}

// The BH's rows of mu, by the threads of one workgroup.
__device__ __forceinline__ void adj_prep_bh(const AdjLin& l, double* __restrict__ mu, size_t cap,
                                            int b0)
{
    if (threadIdx.x < 6) mu[threadIdx.x * cap + b0] = adj_lin(l, threadIdx.x * cap + b0);
}

__global__ __launch_bounds__(FWG) void k_adj_prep(const double* __restrict__ y, AdjLin l,
                                                 double* __restrict__ mu,
                                                 const double* __restrict__ m, Phys P, int nrow,
                                                 ARec* __restrict__ rec,
                                                 double* __restrict__ jd,
                                                 double* __restrict__ rows,
                                                 double* __restrict__ sums,
                                                 unsigned int* __restrict__ ticket)
{
    __shared__ double tot[RV];
    const int row = blockIdx.x * FG + (int)(threadIdx.x >> 6);
    const int p = 1 + row * RB + (int)(threadIdx.x & 63);
    if (row < nrow)
        adj_prep_row(y, l, mu, m, (size_t)P.cap, P.eps2, P.lam, p, p < P.n, 0, rec, jd, rows,
                     row);
    if (blockIdx.x == 0) adj_prep_bh(l, mu, (size_t)P.cap, 0);
    if (last_block(ticket, gridDim.x)) {
        rows_total(rows, 0, nrow, tot);
        if (threadIdx.x < RV) sums[threadIdx.x] = tot[threadIdx.x];
    }
}

// What the VJP of one stage adds its result to (null: nothing), in this
// order: out = ((z0 + z1) + z2) + result.
struct AdjAdd {
    const double *z0, *z1, *z2;
};
__device__ __forceinline__ double adj_add(const AdjAdd& z, size_t i, double r)
{
    return z.z0 ? ((z.z0[i] + z.z1[i]) + z.z2[i]) + r : r;
}

// Stars of one row: the pair kernel's partials (part: S rows of NADJ1 i-side
// sums, then nIb rows of NADJ2 j-side sums, of stride `stride`), the
// separable terms from the sums over all stars, and the star terms.  out_x =
// g_x, out_v = mu_x + g_v (the VJP of the stage function (x, v) -> (v, a)).
// G = FG: the workgroup's waves share the row; G = 1: a row per wave (as
// fin_rows).  Every thread of the workgroup calls it.
template <int G>
__device__ __forceinline__ void adj_fin_row(const ARec* __restrict__ rec,
                                            const double* __restrict__ y,
                                            const double* __restrict__ mu,
                                            const double* __restrict__ m,
                                            const double* __restrict__ part, int S, int nIb,
                                            size_t stride, size_t idx, int p, bool ok, int b0,
                                            const double* __restrict__ sums, AdjAdd z,
                                            double* __restrict__ out, double* __restrict__ rows,
                                            int row, const Phys& P)
{
    const int lane = threadIdx.x & 63;
    const int w = G == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const size_t cap = (size_t)P.cap;
    double g[NADJ1];
#pragma unroll
    for (int k = 0; k < NADJ1; ++k) g[k] = 0.0;
    for (int s = w; s < S; s += G) {
        double L[NADJ1];
#pragma unroll
        for (int k = 0; k < NADJ1; ++k) L[k] = part[(size_t)(s * NADJ1 + k) * stride + idx];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < NADJ1; ++k) g[k] += L[k];
    }
    const double* pj = part + (size_t)S * NADJ1 * stride;
    for (int b = w; b < nIb; b += G) {
        double L[NADJ2];
#pragma unroll
        for (int k = 0; k < NADJ2; ++k) L[k] = pj[(size_t)(b * NADJ2 + k) * stride + idx];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < NADJ2; ++k) g[k] += L[k];
    }
    if (G > 1) {
        __shared__ double sh[G > 1 ? G / 2 : 1][NADJ1][RB];
#pragma unroll
        for (int h = G / 2; h >= 1; h >>= 1) {
            if (w >= h && w < 2 * h)
#pragma unroll
                for (int k = 0; k < NADJ1; ++k) sh[w - h][k][lane] = g[k];
            __syncthreads();
            if (w < h)
#pragma unroll
                for (int k = 0; k < NADJ1; ++k) g[k] += sh[w][k][lane];
            __syncthreads();
        }
        if (w > 0) return;
    }
    double v[RV];
#pragma unroll
    for (int k = 0; k < RV; ++k) v[k] = 0.0;
    if (ok) {
        const ABH B = load_abh(y, mu, m, P.cap, b0);
        const RevU U = rev_uniform(B, P.eps2, P.lam);
        const ARec me = rec[p];
        // the separable terms: the sums over all stars less this one's share
        const RevI I = rev_setup(me, U);
        const RevJ J = rev_jrec(me);
        const RevD D = rev_derive(J, U, me.m);
        RevIAcc ai;
        RevJAcc aj;
        rev_zero(ai);
        rev_zero(aj);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            ai.mv[k] = sums[k] - me.m * I.v[k];
            ai.qs[k] = sums[3 + k] - D.Qd[k];
            aj.t[k] = me.m * (sums[6 + k]
                              - P.lam * (I.Kc * I.v[k] + I.Kd * I.d[k] + I.Ke * I.u[k]));
        }
        aj.ka = me.m * (sums[9] - I.nKa);
        aj.kf = me.m * (sums[10] - I.Kfl);
        aj.kg = me.m * (sums[11] - P.lam * I.Kg);
        double gi[NADJ1], gj[NADJ2];
        rev_ifin(me, U, ai, gi);
        rev_jfin(J, U, aj, gj);
#pragma unroll
        for (int k = 0; k < NADJ1; ++k) g[k] += gi[k];
#pragma unroll
        for (int k = 0; k < NADJ2; ++k) g[k] += gj[k];
        adj_star_grad(me, B, P.eps, P.eps2, P.lam, gi);
#pragma unroll
        for (int k = 0; k < NADJ1; ++k) g[k] += gi[k];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const size_t ix = k * cap + p, iv = (3 + k) * cap + p;
            out[ix] = adj_add(z, ix, g[k]);
            out[iv] = adj_add(z, iv, mu[ix] + g[3 + k]);
            v[k] = g[k];
        }
        v[3] = g[6];
    }
    const double t = wave_sums16(v);
    if ((lane & 3) == 0) hand_over(&rows[(size_t)row * RV + (lane >> 2)], t);
}

// After the last row: the BH at b0, out_x = -(sum of the stars' g_x), out_v =
// mu_x; the m0 derivative of this evaluation goes to gm0[1] and is added to
// gm0[0].
__device__ __forceinline__ void adj_close(const double* __restrict__ rows, int r0, int r1, int b0,
                                          const double* __restrict__ mu, AdjAdd z,
                                          double* __restrict__ out, double* __restrict__ gm0,
                                          size_t cap)
{
    __shared__ double tot[RV];
    rows_total(rows, r0, r1, tot);
    const int k = threadIdx.x;
    if (k < 3) {
        const size_t ix = k * cap + b0, iv = (3 + k) * cap + b0;
        out[ix] = adj_add(z, ix, -tot[k]);
        out[iv] = adj_add(z, iv, mu[ix]);
    }
    if (k == 0) {
        gm0[1] = tot[3];
        gm0[0] += tot[3];
    }
}

template <int G>
__global__ __launch_bounds__(FWG) void k_adj_fin(const ARec* __restrict__ rec,
                                                const double* __restrict__ y,
                                                const double* __restrict__ mu,
                                                const double* __restrict__ m,
                                                const double* __restrict__ part, int S, int nIb,
                                                const double* __restrict__ sums, AdjAdd z,
                                                double* out, double* __restrict__ gm0, int nrow,
                                                double* __restrict__ rows,
                                                unsigned int* __restrict__ ticket, Phys P)
{
    const int row = G == 1 ? (int)blockIdx.x * FG + (int)(threadIdx.x >> 6) : (int)blockIdx.x;
    const int p = 1 + row * RB + (int)(threadIdx.x & 63);
    if (G > 1 || row < nrow)
        adj_fin_row<G>(rec, y, mu, m, part, S, nIb, (size_t)P.cap, (size_t)min(p, P.cap - 1), p,
                       p < P.n, 0, sums, z, out, rows, row, P);
    if (last_block(ticket, gridDim.x)) adj_close(rows, 0, nrow, 0, mu, z, out, gm0, (size_t)P.cap);
}

}  // namespace pn1dev
