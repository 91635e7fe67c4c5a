// pn1_adj.hip -- adjoint of libpn1's force and stage driver (the
// pn1_force_vjp / pn1_adjoint_* entry points).  A translation unit of its
// own: it is built with -ffinite-math-only -fno-signed-zeros so that the
// dual-number arithmetic of the per-star VJP terms drops the zero tangents
// of its seeds at compile time; the forward kernels keep strict IEEE
// semantics in pn1_api.hip.  The O(n^2) pair sums of the VJP run in one
// pass (k_adj_rev, pn1_adj_rev.hpp): a hand-written reverse sweep per pair
// gives both of its sides, the j records rotating through the wave's lanes.
//
// The stage driver (Limit-sticky9.c:841-893) maps a state s = (x, v) to
//   Y1 = s + dt/2 F(s),  Y2 = s + dt/2 F(Y1),  s' = s + dt/6 (F(s) + F(Y1) + F(Y2))
// with F(y) = (y_v, a(y)) (its weights sum to 1/2, as in the reference).
// Its discrete adjoint, for the cotangent L' of s':
//   LY2 = J_F(Y2)^T (dt/6 L')
//   LY1 = J_F(Y1)^T (dt/6 L' + dt/2 LY2)
//   L   = L' + LY2 + LY1 + J_F(s)^T (dt/6 L' + dt/2 LY1)
// where J_F(y)^T (mu_x, mu_v) = (J_a,x^T mu_v, mu_x + J_a,v^T mu_v), and
// d/dm0 collects (d a / d m0)^T mu_v of all three.
//
// pn1_adjoint_forward steps the state with the FP64 kernels and keeps a
// checkpoint every `interval` steps; pn1_adjoint_backward re-runs each
// segment from its checkpoint, keeping every step's s, Y1 and Y2 (the
// stage buffers H1, H2 of the step), then walks it backward with three
// VJPs per step and no further force evaluation.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "pn1_adj_rev.hpp"
#include "pn1_ctx.hpp"
#include "pn1_ens.hpp"

using namespace pn1dev;
using namespace pn1host;

struct pn1_adj {
    int cap = 0;
    double *mu = nullptr, *out = nullptr, *L = nullptr, *LY1 = nullptr, *LY2 = nullptr;
    double *gm0 = nullptr, *sums = nullptr;
    ARec* rec = nullptr;
    double* jd = nullptr;       // the pair kernel's records (RevD), [REVD_F][cap]
    double* rpart = nullptr;    // pair kernel partials, rpart_n doubles
    size_t rpart_n = 0;
    double* ckpt = nullptr;     // nck states of 6 x cap
    double* seg = nullptr;      // per step of a segment: s, Y1, Y2 (6 x cap each)
    int nck_cap = 0, seg_cap = 0;
    // recorded by pn1_adjoint_forward
    bool have_fwd = false;
    int steps = 0, interval = 0;
    unsigned gen = 0;
};

namespace pn1host {

void adj_free(pn1_ctx* c)
{
    pn1_adj* a = c ? c->adj : nullptr;
    if (!a) return;
    void* bufs[] = {a->mu, a->out, a->L, a->LY1, a->LY2, a->gm0, a->sums, a->rec, a->jd, a->rpart,
                    a->ckpt, a->seg};
    for (void* b : bufs)
        if (b) (void)hipFree(b);
    delete a;
    c->adj = nullptr;
}

}  // namespace pn1host

namespace {

template <typename T>
int aalloc(pn1_ctx* c, T** p, size_t count)
{
    if (dev_malloc((void**)p, (count ? count : 1) * sizeof(T)) != hipSuccess) {
        *p = nullptr;
        return seterr(c, PN1_ENOMEM, "hipMalloc of %zu bytes (adjoint) failed", count * sizeof(T));
    }
    return PN1_OK;
}

// Buffers sized for the context's capacity (allocated once).
int adj_get(pn1_ctx* c, pn1_adj** out)
{
    if (!c->adj) {
        pn1_adj* a = new pn1_adj;
        c->adj = a;
        a->cap = c->cap;
        const size_t s6 = 6 * (size_t)c->cap;
        int rc = PN1_OK;
        if (!rc) rc = aalloc(c, &a->mu, s6);
        if (!rc) rc = aalloc(c, &a->out, s6);
        if (!rc) rc = aalloc(c, &a->L, s6);
        if (!rc) rc = aalloc(c, &a->LY1, s6);
        if (!rc) rc = aalloc(c, &a->LY2, s6);
        if (!rc) rc = aalloc(c, &a->gm0, 2);
        if (!rc) rc = aalloc(c, &a->sums, RV);
        if (!rc) rc = aalloc(c, &a->jd, (size_t)REVD_F * c->cap);
        if (!rc) rc = aalloc(c, &a->rec, (size_t)c->cap + 2);
        if (rc) {
            adj_free(c);
            return rc;
        }
    }
    *out = c->adj;
    return PN1_OK;
}

// j chunk L of the single-pass pair kernel for nst stars in nIb blocks of
// 256: whole 64-record tiles, the longest that still gives about
// PN1_ADJ_BLOCKS workgroups (several rounds of the whole device), within
// [64, 2048].  At n = 16385, L = 128 ... 1024 time within 2% of each
// other; at n = 2049, 64-record chunks (a tile per wave, the least there is)
// put twice the workgroups of 128-record ones on the chip (52 -> 32 us).  The partials take ceil(nst / L) * 7 + nIb * 6 rows of cap doubles:
// the j-side rows (one per 256-star block) dominate, ~n^2 / 5.3 bytes.
#ifndef PN1_ADJ_BLOCKS
#define PN1_ADJ_BLOCKS 2048
#endif
int adj_chunk(int nst, int nIb)
{
    const int s0 = std::max(1, (PN1_ADJ_BLOCKS + nIb - 1) / std::max(nIb, 1));
    int L = (nst + s0 - 1) / s0;
    L = (L + 63) / 64 * 64;
    return std::min(std::max(L, 64), 2048);
}

// Rows up to which k_adj_fin's workgroups share a row among their waves (as
// k_fin's).
constexpr int ADJ_FIN_ROWS = 1024;

// out = z + J_F(y)^T mu for the state y (SoA 6 x cap) and the cotangent mu = l
// (z: nothing if null); d/dm0 to gm0[1], added to gm0[0].  FP64.
int enqueue_vjp(pn1_ctx* c, pn1_adj* a, const double* y, const AdjLin& l, const AdjAdd& z,
                double* out, const Phys& P)
{
    int S = 0, nIb = 0;
    hipLaunchKernelGGL(k_adj_prep, dim3((c->nrow + FG - 1) / FG), dim3(FWG), 0, c->st, y, l, a->mu,
                       c->m, P, c->nrow, a->rec, a->jd, c->rows, a->sums, c->ticket);
    if (c->n > 1) {
        // an explicit j split (pn1_set_tuning, pn1_autotune) sets the chunk
        // count, rounded to whole tiles; otherwise the VJP picks its own
        const int nst = c->n - 1;
        const int L = c->jsplit_req > 0 ? ((nst + c->S - 1) / c->S + 63) / 64 * 64
                                        : adj_chunk(nst, c->nIblk);
        S = (nst + L - 1) / L;
        nIb = c->nIblk;
        const size_t need = ((size_t)S * NADJ1 + (size_t)nIb * NADJ2) * (size_t)c->cap;
        if (need > a->rpart_n) {
            if (a->rpart) (void)hipFree(a->rpart);
            a->rpart = nullptr;
            a->rpart_n = 0;
            int rc = aalloc(c, &a->rpart, need);
            if (rc) return rc;
            a->rpart_n = need;
        }
        hipLaunchKernelGGL(k_adj_rev, dim3(S * nIb), dim3(WG), 0, c->st, a->rec, a->jd, y, a->mu,
                           c->m, a->rpart, P, L, S);
    }
    if (c->nrow <= ADJ_FIN_ROWS)
        hipLaunchKernelGGL(k_adj_fin<FG>, dim3(c->nrow), dim3(FWG), 0, c->st, a->rec, y, a->mu,
                           c->m, (const double*)a->rpart, S, nIb, a->sums, z, out, a->gm0,
                           c->nrow, c->rows, c->ticket, P);
    else
        hipLaunchKernelGGL(k_adj_fin<1>, dim3((c->nrow + FG - 1) / FG), dim3(FWG), 0, c->st,
                           a->rec, y, a->mu, c->m, (const double*)a->rpart, S, nIb, a->sums, z,
                           out, a->gm0, c->nrow, c->rows, c->ticket, P);
    HIPCHK(c, hipGetLastError());
    return PN1_OK;
}

// The adjoint runs the FP64 kernels whatever the context's mode.
struct Fp64Scope {
    pn1_ctx* c;
    int mode;
    explicit Fp64Scope(pn1_ctx* cc) : c(cc), mode(cc->mode) { c->mode = PN1_FP64; }
    ~Fp64Scope() { c->mode = mode; }
};

// Stages 1 and 2 of a step written to Y1 and Y2 (6 x cap each) instead of the
// stage states H1 and H2.
template <class C>
struct StageScope {
    C* c;
    double *h1, *h2;
    StageScope(C* cc, double* Y1, double* Y2) : c(cc), h1(cc->H1), h2(cc->H2)
    {
        c->H1 = Y1;
        c->H2 = Y2;
    }
    ~StageScope()
    {
        c->H1 = h1;
        c->H2 = h2;
    }
};

// The first `last` evaluations of a step, the first of them prepared.
int enqueue_stages(pn1_ctx* c, int last, const Phys& P)
{
    for (int stage = 1; stage <= last; ++stage) {
        int rc = enqueue_eval(c, stage, P);
        if (rc) return rc;
    }
    return PN1_OK;
}

}  // namespace

extern "C" {

int pn1_force_vjp(pn1_ctx* c, const double* u, double* gx, double* gv, double* gm0)
{
    int rc;
    if (!ready(c, &rc)) return rc;
    if (!u || !gx || !gv) return seterr(c, PN1_EINVAL, "null argument");
    pn1_adj* a;
    if ((rc = adj_get(c, &a))) return rc;
    const Phys P = make_phys(c);
    if ((rc = put6(c, nullptr, u, a->L, a->gm0, 2))) return rc;
    const AdjLin mu = {a->L, nullptr, 1.0, 0.0};
    if ((rc = enqueue_vjp(c, a, c->X, mu, AdjAdd{}, a->out, P))) return rc;
    double h[2];
    if ((rc = fetch(c, a->out, c->n, gx, gv, a->gm0, 2, h))) return rc;
    if (gm0) *gm0 = h[1];
    return PN1_OK;
}

int pn1_adjoint_forward(pn1_ctx* c, int steps, int interval)
{
    int rc;
    if (!ready(c, &rc)) return rc;
    if (steps < 1 || interval < 1)
        return seterr(c, PN1_EINVAL, "steps (%d) and interval (%d) must be >= 1", steps, interval);
    pn1_adj* a;
    if ((rc = adj_get(c, &a))) return rc;
    // a run that stops below leaves nothing for pn1_adjoint_backward to
    // reverse (its checkpoint buffers may have been replaced)
    a->have_fwd = false;
    const int nck = (steps + interval - 1) / interval;
    const size_t s6 = 6 * (size_t)c->cap;
    if (nck > a->nck_cap) {
        if (a->ckpt) (void)hipFree(a->ckpt);
        a->ckpt = nullptr;
        a->nck_cap = 0;
        if ((rc = aalloc(c, &a->ckpt, (size_t)nck * s6))) return rc;
        a->nck_cap = nck;
    }
    const int seg = std::min(interval, steps);
    if (seg > a->seg_cap) {
        if (a->seg) (void)hipFree(a->seg);
        a->seg = nullptr;
        a->seg_cap = 0;
        if ((rc = aalloc(c, &a->seg, 3 * (size_t)seg * s6))) return rc;
        a->seg_cap = seg;
    }
    Fp64Scope fp64(c);
    drop_graph(c);
    const Phys P = make_phys(c);
    if ((rc = enqueue_prep(c, P))) return rc;
    for (int t = 0; t < steps; ++t) {
        if (t % interval == 0)
            HIPCHK(c, copy6(c->st, a->ckpt + (size_t)(t / interval) * s6, c->X, c->n, c->cap));
        if ((rc = enqueue_stages(c, 3, P))) return rc;
    }
    HIPCHK(c, hipStreamSynchronize(c->st));
    a->have_fwd = true;
    a->steps = steps;
    a->interval = interval;
    a->gen = c->gen;
    return PN1_OK;
}

int pn1_adjoint_backward(pn1_ctx* c, const double* gx, const double* gv, double* gx0,
                         double* gv0, double* gm0)
{
    int rc;
    if (!ready(c, &rc)) return rc;
    if (!gx || !gv || !gx0 || !gv0) return seterr(c, PN1_EINVAL, "null argument");
    pn1_adj* a = c->adj;
    if (!a || !a->have_fwd) return seterr(c, PN1_EINVAL, "no pn1_adjoint_forward run to reverse");
    if (a->gen != c->gen)
        return seterr(c, PN1_EINVAL, "state or parameters changed since pn1_adjoint_forward");
    Fp64Scope fp64(c);
    drop_graph(c);
    const Phys P = make_phys(c);
    const double dt = c->dt;
    const size_t s6 = 6 * (size_t)c->cap;
    if ((rc = put6(c, gx, gv, a->L, a->gm0, 2))) return rc;
    const int nck = (a->steps + a->interval - 1) / a->interval;
    for (int k = nck - 1; k >= 0; --k) {
        const int t0 = k * a->interval, t1 = std::min(a->steps, t0 + a->interval);
        // the segment's states: per step s, Y1 = H1 and Y2 = H2 (the last
        // step runs two stages only: its end state is not needed)
        HIPCHK(c, copy6(c->st, c->X, a->ckpt + (size_t)k * s6, c->n, c->cap));
        if ((rc = enqueue_prep(c, P))) return rc;
        for (int t = t0; t < t1; ++t) {
            double* st = a->seg + 3 * (size_t)(t - t0) * s6;
            HIPCHK(c, copy6(c->st, st, c->X, c->n, c->cap));
            const StageScope<pn1_ctx> keep(c, st + s6, st + 2 * s6);
            if ((rc = enqueue_stages(c, t + 1 < t1 ? 3 : 2, P))) return rc;
        }
        for (int t = t1 - 1; t >= t0; --t) {
            const double* st = a->seg + 3 * (size_t)(t - t0) * s6;
            const AdjLin m2 = {a->L, nullptr, dt / 6.0, 0.0};
            const AdjLin m1 = {a->L, a->LY2, dt / 6.0, dt / 2.0};
            const AdjLin m0 = {a->L, a->LY1, dt / 6.0, dt / 2.0};
            const AdjAdd sum = {a->L, a->LY2, a->LY1};
            if ((rc = enqueue_vjp(c, a, st + 2 * s6, m2, AdjAdd{}, a->LY2, P))) return rc;
            if ((rc = enqueue_vjp(c, a, st + s6, m1, AdjAdd{}, a->LY1, P))) return rc;
            if ((rc = enqueue_vjp(c, a, st, m0, sum, a->L, P))) return rc;
        }
    }
    HIPCHK(c, copy6(c->st, c->X, a->ckpt, c->n, c->cap));    // leave the initial state
    double h[2];
    if ((rc = fetch(c, a->L, c->n, gx0, gv0, a->gm0, 2, h))) return rc;
    if (gm0) *gm0 = h[0];
    return PN1_OK;
}

}  // extern "C"

// =========================================================================
// Ensembles (pn1_ens_force_vjp, pn1_ens_adjoint_*): the same VJP and stage
// adjoint for every cluster at once.  The single-pass pair kernel is a
// persistent launch over the ensemble's own work items (cluster, 256-star
// block, j chunk) and per-XCD queues; each item writes its own partial rows.
// =========================================================================
namespace pn1dev {

// As k_adj_prep, one workgroup per FG rows of a cluster (pblk; crow: its
// rows); it also resets the pair kernel's queues.
__global__ __launch_bounds__(FWG) void k_ens_adj_prep(const double* __restrict__ y, AdjLin l,
                                                     double* __restrict__ mu,
                                                     const double* __restrict__ m,
                                                     const int* __restrict__ coff,
                                                     const int* __restrict__ crow,
                                                     const EBlk* __restrict__ pblk, int npblk,
                                                     Phys P,
                                                     ARec* __restrict__ rec,
                                                     double* __restrict__ jd,
                                                     double* __restrict__ rows,
                                                     double* __restrict__ sums,
                                                     unsigned int* __restrict__ ticket,
                                                     unsigned int* __restrict__ counter)
{
    __shared__ double tot[RV];
    const int wg = ens_block();
    if (wg == 0 && threadIdx.x < NXCD) counter[threadIdx.x] = 0u;
    if (wg >= npblk) return;
    const EBlk b = pblk[wg];
    const int off = coff[b.c], nst = coff[b.c + 1] - off - 1;
    const int r0 = crow[b.c], r1 = crow[b.c + 1];
    const int row = r0 + b.first / RB + (int)(threadIdx.x >> 6);
    const int li = b.first + (int)threadIdx.x;
    if (row < r1)
        adj_prep_row(y, l, mu, m, (size_t)P.cap, P.eps2, P.lam, off + 1 + li, li < nst, off, rec,
                     jd, rows, row);
    if (b.first == 0) adj_prep_bh(l, mu, (size_t)P.cap, off);
    if (last_block(ticket + b.c, (unsigned)((r1 - r0 + FG - 1) / FG))) {
        rows_total(rows, r0, r1, tot);
        if (threadIdx.x < RV) sums[(size_t)b.c * RV + threadIdx.x] = tot[threadIdx.x];
    }
}

// Persistent single-pass pair kernel over the ensemble's work items.  Item
// (cluster c, block ib, chunk s): stars off + 1 + ib*WG + lane, records
// [j0, j1).  The partials of cluster c start at apart + aoff[c], rows of
// stride nst: i side (s*NADJ1 + k), s < S_c; then j side
// (S_c*NADJ1 + ib*NADJ2 + k).  Every item writes its own rows.
__global__ __launch_bounds__(WG) void k_ens_adj_rev(const ARec* __restrict__ rec,
                                                   const double* __restrict__ jd,
                                                   const double* __restrict__ y,
                                                   const double* __restrict__ mu,
                                                   const double* __restrict__ m,
                                                   double* __restrict__ apart,
                                                   const long long* __restrict__ aoff,
                                                   const EItem* __restrict__ items,
                                                   unsigned int* __restrict__ counter,
                                                   const int* __restrict__ qoff, Phys P, int L)
{
    int q = 0;
    for (;;) {
        const int it = ens_take(counter, qoff, q);
        if (it < 0) break;
        const EItem w = items[it];
        const int nst = w.nst;
        const int li = w.ib * WG + (int)threadIdx.x;
        const bool iok = li < nst;
        const bool live = w.ib * WG + (__builtin_amdgcn_readfirstlane((int)threadIdx.x) & ~63) < nst;
        const RevU U = rev_uniform(load_abh(y, mu, m, P.cap, w.off), P.eps2, P.lam);
        const int S = ens_nchunks(nst, L), s = (w.j0 - w.off - 1) / L;
        double* base = apart + aoff[w.c];
        double* pj = base + ((size_t)S * NADJ1 + (size_t)w.ib * NADJ2) * nst;
        double g[NADJ1];
        rev_chunk(rec, jd, (size_t)P.cap, U, w.off + 1 + (iok ? li : nst - 1), iok, live, w.j0,
                  w.j1, g, [&](int j, const double (&gj)[NADJ2]) {
#pragma unroll
                      for (int k = 0; k < NADJ2; ++k)
                          pj[(size_t)k * nst + (j - w.off - 1)] = gj[k];
                  });
        if (iok) {
#pragma unroll
            for (int k = 0; k < NADJ1; ++k) base[((size_t)s * NADJ1 + k) * nst + li] = g[k];
        }
    }
}

// As k_adj_fin, one workgroup per row (G = FG, blk the row table) or per FG
// rows of a cluster (G = 1, blk = pblk); gm0[2c], gm0[2c + 1] of cluster c.
template <int G>
__global__ __launch_bounds__(FWG) void k_ens_adj_fin(const ARec* __restrict__ rec,
                                                    const double* __restrict__ y,
                                                    const double* __restrict__ mu,
                                                    const double* __restrict__ m,
                                                    const int* __restrict__ coff,
                                                    const int* __restrict__ crow,
                                                    const EBlk* __restrict__ blk, int n,
                                                    const double* __restrict__ apart,
                                                    const long long* __restrict__ aoff,
                                                    const double* __restrict__ sums, AdjAdd z,
                                                    double* out, double* __restrict__ gm0,
                                                    double* __restrict__ rows,
                                                    unsigned int* __restrict__ ticket, Phys P,
                                                    int L)
{
    const int wg = ens_block();
    if (wg >= n) return;
    const EBlk b = blk[wg];
    const int off = coff[b.c], nst = coff[b.c + 1] - off - 1;
    const int r0 = crow[b.c], r1 = crow[b.c + 1];
    const int li = b.first + (int)(G == 1 ? threadIdx.x : threadIdx.x & 63);
    const int row = r0 + li / RB;
    if (G > 1 || row < r1)
        adj_fin_row<G>(rec, y, mu, m, apart + aoff[b.c], nst > 0 ? ens_nchunks(nst, L) : 0,
                       (nst + WG - 1) / WG, (size_t)nst, (size_t)max(min(li, nst - 1), 0),
                       off + 1 + li, li < nst, off, sums + (size_t)b.c * RV, z, out, rows, row,
                       P);
    if (last_block(ticket + b.c, (unsigned)(G == 1 ? (r1 - r0 + FG - 1) / FG : r1 - r0)))
        adj_close(rows, r0, r1, off, mu, z, out, gm0 + 2 * (size_t)b.c, (size_t)P.cap);
}

}  // namespace pn1dev

struct pn1_ens_adj {
    double *mu = nullptr, *out = nullptr, *L = nullptr, *LY1 = nullptr, *LY2 = nullptr;
    double *gm0 = nullptr, *sums = nullptr;
    ARec* rec = nullptr;
    double* jd = nullptr;         // the pair kernel's records (RevD), [REVD_F][cap]
    double* ckpt = nullptr;
    double* seg = nullptr;        // per step of a segment: s, Y1, Y2 (6 x cap each)
    int nck_cap = 0, seg_cap = 0;
    int grid = 0;                 // resident workgroups of k_ens_adj_rev
    double* apart = nullptr;      // pair kernel partials, apart_n doubles
    size_t apart_n = 0;
    long long* aoff = nullptr;    // per-cluster offsets into apart (capc)
    unsigned tab_gen = 0;         // (gen, L) the offsets were made for
    int tab_L = -1;
    bool have_fwd = false;
    int steps = 0, interval = 0;
    unsigned gen = 0;
};

namespace pn1host {

void ens_adj_free(pn1_ens* e)
{
    pn1_ens_adj* a = e ? e->adj : nullptr;
    if (!a) return;
    void* bufs[] = {a->mu, a->out, a->L, a->LY1, a->LY2, a->gm0, a->sums, a->rec, a->jd,
                    a->ckpt, a->seg, a->apart, a->aoff};
    for (void* b : bufs)
        if (b) (void)hipFree(b);
    delete a;
    e->adj = nullptr;
}

}  // namespace pn1host

namespace {

template <typename T>
int ealloc_adj(pn1_ens* e, T** p, size_t count)
{
    if (dev_malloc((void**)p, (count ? count : 1) * sizeof(T)) != hipSuccess) {
        *p = nullptr;
        return eerr(e, PN1_ENOMEM, "hipMalloc of %zu bytes (adjoint) failed", count * sizeof(T));
    }
    return PN1_OK;
}

template <typename K>
int adj_resident_grid(pn1_ens* e, K kernel, int* out)
{
    int per_cu = 0, dev = 0;
    hipDeviceProp_t prop;
    EHIPCHK(e, hipGetDevice(&dev));
    EHIPCHK(e, hipGetDeviceProperties(&prop, dev));
    EHIPCHK(e, hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, WG, 0));
    *out = (per_cu > 0 ? per_cu : 1) * prop.multiProcessorCount;
    return PN1_OK;
}

int ens_adj_get(pn1_ens* e, pn1_ens_adj** out)
{
    if (!e->adj) {
        pn1_ens_adj* a = new pn1_ens_adj;
        e->adj = a;
        const size_t s6 = 6 * (size_t)e->cap;
        int rc = PN1_OK;
        if (!rc) rc = ealloc_adj(e, &a->mu, s6);
        if (!rc) rc = ealloc_adj(e, &a->out, s6);
        if (!rc) rc = ealloc_adj(e, &a->L, s6);
        if (!rc) rc = ealloc_adj(e, &a->LY1, s6);
        if (!rc) rc = ealloc_adj(e, &a->LY2, s6);
        if (!rc) rc = ealloc_adj(e, &a->gm0, 2 * (size_t)e->capc);
        if (!rc) rc = ealloc_adj(e, &a->sums, (size_t)RV * e->capc);
        if (!rc) rc = ealloc_adj(e, &a->jd, (size_t)REVD_F * e->cap);
        if (!rc) rc = ealloc_adj(e, &a->rec, (size_t)e->cap + 2);
        if (!rc) rc = ealloc_adj(e, &a->aoff, (size_t)e->capc);
        if (!rc) rc = adj_resident_grid(e, k_ens_adj_rev, &a->grid);
        if (rc) {
            ens_adj_free(e);
            return rc;
        }
    }
    pn1_ens_adj* a = e->adj;
    if (int rc = ens_items(e)) return rc;
    if (a->tab_L != e->L || a->tab_gen != e->gen) {   // partial layout of the clusters
        std::vector<long long> aoff(e->nc > 0 ? e->nc : 1, 0);
        size_t tot = 0;
        for (int c = 0; c < e->nc; ++c) {
            const int nst = e->off_h[c + 1] - e->off_h[c] - 1;
            aoff[c] = (long long)tot;
            if (nst > 0)
                tot += ((size_t)((nst + e->L - 1) / e->L) * NADJ1 +
                        (size_t)((nst + WG - 1) / WG) * NADJ2) * (size_t)nst;
        }
        if (tot > a->apart_n) {
            if (a->apart) (void)hipFree(a->apart);
            a->apart = nullptr;
            a->apart_n = 0;
            int rc = ealloc_adj(e, &a->apart, tot);
            if (rc) return rc;
            a->apart_n = tot;
        }
        if (e->nc > 0)
            EHIPCHK(e, hipMemcpyAsync(a->aoff, aoff.data(), e->nc * sizeof(long long),
                                      hipMemcpyHostToDevice, e->st));
        EHIPCHK(e, hipStreamSynchronize(e->st));
        a->tab_L = e->L;
        a->tab_gen = e->gen;
    }
    *out = a;
    return PN1_OK;
}

int ens_enqueue_vjp(pn1_ens* e, pn1_ens_adj* a, const double* y, const AdjLin& l,
                    const AdjAdd& z, double* out, const Phys& P)
{
    hipLaunchKernelGGL(k_ens_adj_prep, ens_grid(e->npblk), dim3(FWG), 0, e->st, y, l, a->mu, e->m,
                       e->coff, e->crow, e->pblk, e->npblk, P, a->rec, a->jd, e->rows, a->sums, e->ticket,
                       e->counter);
    if (e->nitems)
        hipLaunchKernelGGL(k_ens_adj_rev, dim3(std::min(a->grid, e->nitems)), dim3(WG), 0, e->st,
                           a->rec, a->jd, y, a->mu, e->m, a->apart, a->aoff, e->items,
                           e->counter, e->qoff, P, e->L);
    if (e->nrow <= ADJ_FIN_ROWS)
        hipLaunchKernelGGL(k_ens_adj_fin<FG>, dim3(e->nrow), dim3(FWG), 0, e->st, a->rec, y, a->mu,
                           e->m, e->coff, e->crow, e->row, e->nrow, (const double*)a->apart, a->aoff,
                           a->sums, z, out, a->gm0, e->rows, e->ticket, P, e->L);
    else
        hipLaunchKernelGGL(k_ens_adj_fin<1>, ens_grid(e->npblk), dim3(FWG), 0, e->st, a->rec, y,
                           a->mu, e->m, e->coff, e->crow, e->pblk, e->npblk,
                           (const double*)a->apart, a->aoff,
                           a->sums, z, out, a->gm0, e->rows, e->ticket, P, e->L);
    EHIPCHK(e, hipGetLastError());
    return PN1_OK;
}

// Fetches src (6 x cap) to ox, ov and value `which` of each cluster's gm0 pair.
int ens_get(pn1_ens* e, pn1_ens_adj* a, const double* src, double* ox, double* ov, int which,
            double* gm0)
{
    std::vector<double> h(2 * (size_t)e->nc);
    const int rc = ens_fetch(e, src, ox, ov, a->gm0, h.size(), h.data());
    if (rc) return rc;
    for (int c = 0; gm0 && c < e->nc; ++c) gm0[c] = h[2 * (size_t)c + which];
    return PN1_OK;
}

struct EnsFp64Scope {
    pn1_ens* e;
    int mode;
    explicit EnsFp64Scope(pn1_ens* ee) : e(ee), mode(ee->mode) { e->mode = PN1_FP64; }
    ~EnsFp64Scope() { e->mode = mode; }
};

int ens_stages(pn1_ens* e, int last, const Phys& P)
{
    for (int stage = 1; stage <= last; ++stage) {
        int rc = ens_enqueue_eval(e, stage, P);
        if (rc) return rc;
    }
    return PN1_OK;
}

}  // namespace

extern "C" {

int pn1_ens_force_vjp(pn1_ens* e, const double* u, double* gx, double* gv, double* gm0)
{
    int rc;
    if (!ens_force_ready(e, &rc)) return rc;
    if (!u || !gx || !gv) return eerr(e, PN1_EINVAL, "null argument");
    pn1_ens_adj* a;
    if ((rc = ens_adj_get(e, &a))) return rc;
    const Phys P = ens_phys(e);
    if ((rc = ens_put6(e, nullptr, u, a->L, a->gm0, 2 * (size_t)e->nc))) return rc;
    const AdjLin mu = {a->L, nullptr, 1.0, 0.0};
    if ((rc = ens_enqueue_vjp(e, a, e->X, mu, AdjAdd{}, a->out, P))) return rc;
    return ens_get(e, a, a->out, gx, gv, 1, gm0);
}

int pn1_ens_adjoint_forward(pn1_ens* e, int steps, int interval)
{
    int rc;
    if (!ens_force_ready(e, &rc)) return rc;
    if (steps < 1 || interval < 1)
        return eerr(e, PN1_EINVAL, "steps (%d) and interval (%d) must be >= 1", steps, interval);
    pn1_ens_adj* a;
    if ((rc = ens_adj_get(e, &a))) return rc;
    a->have_fwd = false;                 // as in pn1_adjoint_forward
    const int nck = (steps + interval - 1) / interval;
    const size_t s6 = 6 * (size_t)e->cap;
    if (nck > a->nck_cap) {
        if (a->ckpt) (void)hipFree(a->ckpt);
        a->ckpt = nullptr;
        a->nck_cap = 0;
        if ((rc = ealloc_adj(e, &a->ckpt, (size_t)nck * s6))) return rc;
        a->nck_cap = nck;
    }
    const int seg = std::min(interval, steps);
    if (seg > a->seg_cap) {
        if (a->seg) (void)hipFree(a->seg);
        a->seg = nullptr;
        a->seg_cap = 0;
        if ((rc = ealloc_adj(e, &a->seg, 3 * (size_t)seg * s6))) return rc;
        a->seg_cap = seg;
    }
    EnsFp64Scope fp64(e);
    edrop_graph(e);
    const Phys P = ens_phys(e);
    if ((rc = ens_enqueue_prep(e, P))) return rc;
    for (int t = 0; t < steps; ++t) {
        if (t % interval == 0)
            EHIPCHK(e, copy6(e->st, a->ckpt + (size_t)(t / interval) * s6, e->X, e->n, e->cap));
        if ((rc = ens_stages(e, 3, P))) return rc;
    }
    EHIPCHK(e, hipStreamSynchronize(e->st));
    a->have_fwd = true;
    a->steps = steps;
    a->interval = interval;
    a->gen = e->gen;
    return PN1_OK;
}

int pn1_ens_adjoint_backward(pn1_ens* e, const double* gx, const double* gv, double* gx0,
                             double* gv0, double* gm0)
{
    int rc;
    if (!ens_force_ready(e, &rc)) return rc;
    if (!gx || !gv || !gx0 || !gv0) return eerr(e, PN1_EINVAL, "null argument");
    pn1_ens_adj* a = e->adj;
    if (!a || !a->have_fwd)
        return eerr(e, PN1_EINVAL, "no pn1_ens_adjoint_forward run to reverse");
    if (a->gen != e->gen)
        return eerr(e, PN1_EINVAL, "state or parameters changed since pn1_ens_adjoint_forward");
    if ((rc = ens_adj_get(e, &a))) return rc;
    EnsFp64Scope fp64(e);
    edrop_graph(e);
    const Phys P = ens_phys(e);
    const double dt = e->dt;
    const size_t s6 = 6 * (size_t)e->cap;
    if ((rc = ens_put6(e, gx, gv, a->L, a->gm0, 2 * (size_t)e->nc))) return rc;
    const int nck = (a->steps + a->interval - 1) / a->interval;
    for (int k = nck - 1; k >= 0; --k) {
        const int t0 = k * a->interval, t1 = std::min(a->steps, t0 + a->interval);
        EHIPCHK(e, copy6(e->st, e->X, a->ckpt + (size_t)k * s6, e->n, e->cap));
        if ((rc = ens_enqueue_prep(e, P))) return rc;
        for (int t = t0; t < t1; ++t) {
            double* st = a->seg + 3 * (size_t)(t - t0) * s6;
            EHIPCHK(e, copy6(e->st, st, e->X, e->n, e->cap));
            const StageScope<pn1_ens> keep(e, st + s6, st + 2 * s6);
            if ((rc = ens_stages(e, t + 1 < t1 ? 3 : 2, P))) return rc;
        }
        for (int t = t1 - 1; t >= t0; --t) {
            const double* st = a->seg + 3 * (size_t)(t - t0) * s6;
            const AdjLin m2 = {a->L, nullptr, dt / 6.0, 0.0};
            const AdjLin m1 = {a->L, a->LY2, dt / 6.0, dt / 2.0};
            const AdjLin m0 = {a->L, a->LY1, dt / 6.0, dt / 2.0};
            const AdjAdd sum = {a->L, a->LY2, a->LY1};
            if ((rc = ens_enqueue_vjp(e, a, st + 2 * s6, m2, AdjAdd{}, a->LY2, P))) return rc;
            if ((rc = ens_enqueue_vjp(e, a, st + s6, m1, AdjAdd{}, a->LY1, P))) return rc;
            if ((rc = ens_enqueue_vjp(e, a, st, m0, sum, a->L, P))) return rc;
        }
    }
    EHIPCHK(e, copy6(e->st, e->X, a->ckpt, e->n, e->cap));  // leave the initial state
    return ens_get(e, a, a->L, gx0, gv0, 0, gm0);
}

}  // extern "C"
