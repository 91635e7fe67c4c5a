// pn1_api.hip -- host side of libpn1: the context API, the three legacy
// shapes of Limit-sticky9 (force, energy, initial_energy), the autotuner and,
// through pn1_ens.inc, the ensemble API.  The adjoint is in pn1_adj.hip, the
// launches of the mixed-form pair kernels in pn1_pair32.hip.
//
// Device layout (FP64 SoA, stride cap, particle 0 = BH):
//   X[6][cap]   state at the start of a step (x, y, z, vx, vy, vz)
//   Y[6][cap]   stage input (the reference's x1, v1)
//   H1, H2      stage states 1 and 2 (the reference's hx[1..2], hv[1..2])
//   m[cap], acc[3][cap]
//   j64[3][cap + 2], j32[cap + 2]   per-evaluation j-records (AoS)
//   part        pair partials: FP64 [S][16][cap]; mixed [S][16 + 3][cap] floats
//               (the sums, then the Kahan compensations of the Newtonian sums)
// Device memory is allocated by pn1_create, and grown by pn1_upload,
// pn1_set_tuning and pn1_autotune (the partial sums follow the j split) and
// by the first adjoint call; pn1_force, pn1_energy and pn1_step only launch
// kernels and copy results.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <utility>
#include <vector>

#include "pn1.h"
#include "pn1_ctx.hpp"
#include "pn1_ens.hpp"
#include "pn1_ens_kernels.hpp"
#include "pn1_io.hpp"
#include "pn1_kernels.hpp"
#include "pn1_pair32.hpp"

using namespace pn1dev;

namespace pn1host {

int seterr(pn1_ctx* c, int code, const char* fmt, ...)
{
    if (c) {
        va_list ap;
        va_start(ap, fmt);
        vsnprintf(c->err, sizeof c->err, fmt, ap);
        va_end(ap);
    }
    return code;
}

template <typename T>
int dalloc(pn1_ctx* c, T** p, size_t count)
{
    if (dev_malloc((void**)p, count * sizeof(T)) != hipSuccess) {
        *p = nullptr;
        return seterr(c, PN1_ENOMEM, "hipMalloc of %zu bytes failed", count * sizeof(T));
    }
    return PN1_OK;
}

Phys make_phys(const pn1_ctx* c)
{
    Phys P;
    P.eps = c->eps;
    P.eps2 = c->eps * c->eps;
    P.lam = 1.0 / (c->c * c->c);
    P.dt = c->dt;
    P.m0 = c->m0;
    P.ws = 1.0 / std::sqrt(P.eps2);
    P.mmax = c->mmax;
    P.eps2f = (float)P.eps2;
    P.m0f = (float)c->m0;
    P.n = c->n;
    P.cap = c->cap;
    return P;
}

// The mixed form's BH-close threshold for stars up to dmax from the BH (see
// PN1_FLAG_ETA): tauf = eta / (6 u D) with D = 2 dmax, room for the stars to
// move away before the next upload.
double flag_threshold(double dmax)
{
    if (!(dmax > 0.0)) return HUGE_VAL;
    return PN1_FLAG_ETA / (6.0 * 0x1p-24 * 2.0 * dmax);
}

// j split of the 256-star kernels where none is set explicitly (i shards):
// many short rounds of workgroups, chunks of at least 64 records.
int auto_split(int nst)
{
    const int nib = nst > 0 ? (nst + WG - 1) / WG : 0;
    int S = 1;
    while (S < 128 && (long)S * nib < 32768 && (nst + 2 * S - 1) / (2 * S) >= 64) S *= 2;
    return nst > 0 && S > nst ? nst : S;
}

// Partials per star of the automatic plan: from 8192 stars on the tapered
// split's 24 (16 long chunks and 8 short ones), below 16, fewer while a
// wave's part would hold fewer than 4 records.  Short parts balance the launch
// and fill the chip, partials cost k_fin.  Measured on MI355X (one evaluation,
// FP64 / mixed, us; 24 is the tapered one):
//   slots       4     8          16           24           32         64
//   n = 1025    25/28 18.6/22.7  18.0/19.7                 21.5/22.4  30/28
//   n = 2049    35/41 23.3/28.7  23.5/23.7                 27/26      37/34
//   n = 10241         178/128    177/111      178/108      182/113    201/130
//   n = 131073                   24850/12860  24808/12715
// Above 2^22 stars the rows alone are over a hundred workgroups per CU, and
// the split only bounds the partials (128 bytes each): at most 2^26 (8.6 GB),
// while a star has more than one; with one, up to 34 GB at 2^28 stars.  Just
// below 2^22 stars the 24 are 12.9 GB.
int auto_slots(int nst)
{
    if (nst >= 8192 && nst < (1 << 22)) return TLONG + TSHORT;
    int s = TLONG;
    while (s > 1 && (nst < 4 * s * PW || (long)nst * s > (1L << 26))) s >>= 1;
    return s;
}

// Partials per star of an explicit split in S chunks where the row kernels take
// it, else 0: from 2 chunks on (one stays one serial sum per star, as an
// ensemble's unsplit chunk is) to 32, as far as a launch holds them, in up to
// 16 chunks of PW parts.  Measured on MI355X, evaluation with the 256-star
// kernels' S chunks / with these, FP64 and mixed, us:
//   n = 129, S = 2    24.9 / 15.8  31.6 / 20.5
//   n = 1025, S = 16  28.9 / 18.9  31.7 / 20.9
//   n = 4097, S = 32  67.0 / 44.6  96.8 / 37.4
//   n = 16384, S = 32  429 / 418    324 / 241
int explicit_slots(int S, int nst)
{
    if (S < 2 || S > 32) return 0;
    const int s = std::min(S, TLONG);
    return (long)s * ((nst + RB - 1) / RB) <= (1L << 22) ? s : 0;
}

// Launch plan of the pair kernels for the current n.
void plan(pn1_ctx* c)
{
    const int nst = c->n - 1;
    c->nrow = nst > 0 ? (nst + RB - 1) / RB : 1;
    c->nIblk = nst > 0 ? (nst + WG - 1) / WG : 0;
    c->slots = 0;
    if (c->jsplit_req > 0) {
        c->S = std::max(1, std::min(c->jsplit_req, std::max(nst, 1)));
        if (c->variant_req < 0 && nst > 0) c->slots = explicit_slots(c->S, nst);
    } else if (c->variant_req >= 0 || nst < 1) {
        c->S = auto_split(nst);
    } else {
        c->slots = auto_slots(nst);
        c->S = c->slots * PW;
    }
    c->tile = c->tile_req > 0 ? (c->tile_req < 2 ? 2 : c->tile_req) : 64;
}

// Bytes of pair partials of `slots` chunks per star (0: the plan's).
size_t part_need(const pn1_ctx* c, int slots = 0)
{
    const size_t cap = (size_t)c->cap;
    const size_t S = (size_t)(slots > 0 ? slots : c->slots ? c->slots : c->S);
    size_t need = S * NACC * cap * sizeof(double);
    const size_t need32 = S * MROWS * cap * sizeof(float);
    if (need32 > need) need = need32;
    return need;
}

// Partial-sum buffer for `slots` chunks per star (default: the plan's).  The
// new buffer is allocated before the old one is freed: if the allocation
// is refused, the old buffer stays (ready() then refuses launches of a
// plan it does not cover).
int ensure_part(pn1_ctx* c, int slots = 0)
{
    const size_t need = part_need(c, slots);
    if (need <= c->part_bytes) return PN1_OK;
    void* p = nullptr;
    if (dev_malloc(&p, need) != hipSuccess)
        return seterr(c, PN1_ENOMEM, "hipMalloc of %zu bytes for pair partials failed", need);
    drop_graph(c);                      // a captured step holds the old buffer
    if (c->part) (void)hipFree(c->part);
    c->part = p;
    c->part_bytes = need;
    return PN1_OK;
}

// Plan and partials of the current n.  Where the automatic plan's partials are
// refused (a capacity far above n: they are laid out by capacity), the
// 256-star kernels' split takes its place, which at large n needs fewer.
int plan_parts(pn1_ctx* c)
{
    plan(c);
    const int rc = ensure_part(c);
    if (!rc || !c->slots || c->jsplit_req > 0) return rc;
    c->slots = 0;
    c->S = auto_split(c->n - 1);
    return ensure_part(c);
}

// Kernel form in use: the requested one, or per mode the faster one
// measured at n = 131073: one record at a time in both modes (the mixed
// kernel then fits 8 waves per SIMD).
int kernel_variant(const pn1_ctx* c)
{
    if (c->variant_req >= 0) return c->mode == PN1_MIXED ? c->variant_req : (c->variant_req & 1);
    return 0;
}

// Whether the mixed pair kernel combines four chunks per workgroup
// (k_pair32q, variant bit 2, splits into a multiple of 4 chunks): a quarter
// of the partial-sum traffic, at ~1.6% more pair-kernel time than one chunk
// per 256-thread workgroup (k_pair32) at n = 131073 on MI355X.
bool quad_pairs(const pn1_ctx* c, int S)
{
    return c->mode == PN1_MIXED && S >= QSUB && S % QSUB == 0 && (kernel_variant(c) & 4);
}

// Partials per star of a launch of the 256-star kernels split in S chunks.
int part_slots(const pn1_ctx* c, int S) { return quad_pairs(c, S) ? S / QSUB : S; }

// The plan's.
int plan_slots(const pn1_ctx* c) { return c->slots ? c->slots : part_slots(c, c->S); }

// Workgroups of a pair launch over nib i blocks with `slots` chunks each
// (map_block's arrangement when slots divides 8).
int pair_grid(int slots, int nib)
{
    if (slots <= 8 && 8 % slots == 0) return 8 * ((nib + 8 / slots - 1) / (8 / slots));
    return slots * nib;
}

void drop_graph(pn1_ctx* c)
{
    if (c->gexec) (void)hipGraphExecDestroy(c->gexec);
    c->gexec = nullptr;
}

bool ready(pn1_ctx* c, int* rc)
{
    if (!c) {
        *rc = PN1_EINVAL;
        return false;
    }
    if (!c->have_state) {
        *rc = seterr(c, PN1_EINVAL, "no state uploaded");
        return false;
    }
    if (c->part_bytes < part_need(c)) {
        *rc = seterr(c, PN1_ENOMEM, "the pair partials (%zu bytes) do not cover the launch plan "
                     "(%zu bytes): an earlier allocation was refused", c->part_bytes,
                     part_need(c));
        return false;
    }
    if (hipSetDevice(c->dev) != hipSuccess) {
        *rc = seterr(c, PN1_EDEVICE, "hipSetDevice(%d) failed", c->dev);
        return false;
    }
    *rc = PN1_OK;
    return true;
}

// ---- one force evaluation (+ stage update) ------------------------------
// The records and hard stars of a step's evaluations are each in a buffer of
// their own: evaluation `stage` reads buffer eval_buf(stage) while its k_fin
// writes that of the next one, next_buf(stage).
int eval_buf(int stage) { return stage <= 1 ? 0 : stage - 1; }
int next_buf(int stage) { return stage % 3; }
size_t rows_of(size_t cap) { return (cap + RB - 1) / RB + 1; }
JRec64* rec_buf(const pn1_ctx* c, int k) { return c->j64 + (size_t)k * ((size_t)c->cap + 2); }
unsigned long long* hard_buf(const pn1_ctx* c, int k)
{
    return c->hmask + (size_t)k * rows_of((size_t)c->cap);
}

// For k_prep, or the k_fin of an evaluation.  ticket false: the sums over the
// rows are not needed (an i shard).
RowBufs row_bufs(const pn1_ctx* c, int stage = 0, bool ticket = true)
{
    RowBufs R;
    R.rows = c->rows;
    R.fmask = c->fmask;
    R.hmask = hard_buf(c, eval_buf(stage));
    R.hnext = hard_buf(c, next_buf(stage));
    R.gs = c->gs;
    R.flist = c->flist;
    R.fn = c->fn;
    R.ticket = ticket ? c->ticket : nullptr;
    R.clear = nullptr;
    return R;
}

// The mixed form's prep inputs (FP64 form: none).
MixPrep mix_prep(const pn1_ctx* c, const Phys& P)
{
    MixPrep M;
    const bool mixed = c->mode == PN1_MIXED;
    M.j32 = mixed ? c->j32 : nullptr;
    M.thr = mixed ? c->thr : nullptr;
    M.mmax = mixed ? c->mmax : 0.0;
    M.tauf = mixed ? c->tauf : 0.0;
    M.lam = mixed ? P.lam : 0.0;
    return M;
}

// k_fin's form: a workgroup per row up to FIN_ROWS rows, per FG rows above (see
// fin_rows); per group of 16 stars where few rows have many partials each.
// Measured on MI355X, evaluation with a workgroup per row / per group, FP64
// and mixed, us:
//   n = 33 (1 partial)  11.3 / 12.2  14.7 / 16.1
//   n = 257 (8)         14.4 / 13.4  17.5 / 16.6
//   n = 1025 (16)       17.6 / 16.0  19.5 / 19.6
//   n = 2049 (16)       23.6 / 23.2  23.7 / 24.0
//   n = 8193 (24)       120.4 / 123.4  77.9 / 84.5
constexpr int FIN_ROWS = 1024, FIN_SUB = 16;
bool fin_sub(int nst, int nrow, int slots) { return nst > 0 && nrow <= FIN_SUB && slots >= FG; }

// Stars i0 .. i1 - 1 (all: every star and the BH), `slots` partials each; rowk:
// by the row kernels.
template <int MODE, int STAGE>
void launch_fin(pn1_ctx* c, const double* in, const Phys& P, int slots, int i0, int i1, bool all,
                bool rowk)
{
    FinBufs F;
    F.in = in;
    F.X = c->X;
    F.Y = c->Y;
    F.H1 = c->H1;
    F.H2 = c->H2;
    F.m = c->m;
    F.acc = c->acc;
    F.kr = c->kr;
    F.xr = c->xr;
    F.hp = rowk && c->nrow <= HROWS ? c->hpart : nullptr;
    F.j64 = rec_buf(c, eval_buf(STAGE));
    F.jnext = rec_buf(c, next_buf(STAGE));
    const int row0 = (i0 - 1) / RB, rows = std::max(1, (i1 - i0 + RB - 1) / RB);
    const RowBufs R = row_bufs(c, STAGE, all);
    auto launch = [&](auto kernel, int wgs) {
        hipLaunchKernelGGL(kernel, dim3(wgs), dim3(FWG), 0, c->st, F, R, (const void*)c->part,
                           slots, mix_prep(c, P), P, row0, i1, c->nrow);
    };
    if (fin_sub(c->n - 1, c->nrow, slots))
        launch(k_fin<MODE, STAGE, FG, 4>, 4 * rows);
    else if (c->nrow <= FIN_ROWS)
        launch(k_fin<MODE, STAGE, FG, 1>, rows);
    else
        launch(k_fin<MODE, STAGE, 1, 1>, (rows + FG - 1) / FG);
}

// The pair kernel over i blocks ib0 .. ib0 + nib - 1 against every star,
// with the j range split in S chunks.  ts (mixed form): also accumulate the
// sums behind the stars' cancellation ratios.
void launch_pair(pn1_ctx* c, const JRec64* j64, const double* in, const Phys& P, int ib0, int nib,
                 int S, bool ts)
{
    const bool mixed = c->mode == PN1_MIXED;
    const dim3 g(pair_grid(S, nib)), blk(WG);
    const int variant = kernel_variant(c);
    if (mixed) {
        launch_pair32(c, j64, in, P, ib0, nib, S, pair32_form(variant, ts, c->eqm));
    } else if (variant & 1) {
        hipLaunchKernelGGL(k_pair64<1>, g, blk, 0, c->st, j64, in, (double*)c->part, P, S, nib,
                           ib0);
    } else {
        hipLaunchKernelGGL(k_pair64<0>, g, blk, 0, c->st, j64, in, (double*)c->part, P, S, nib,
                           ib0);
    }
}

// The same by the row kernels, rows row0 .. row0 + nrow - 1, the plan's slots,
// with the records (and hard stars) of buffer k.
void launch_pairw(pn1_ctx* c, int k, const double* in, const Phys& P, int row0, int nrow, bool ts)
{
    const JRec64* j64 = rec_buf(c, k);
    if (c->mode == PN1_MIXED)
        launch_pair32w(c, j64, hard_buf(c, k), in, P, c->slots, row0, nrow, ts);
    else
        hipLaunchKernelGGL(k_pair64w, dim3(c->slots * nrow), dim3(PW * RB), 0, c->st, j64, in,
                           (double*)c->part, P, c->slots, nrow, c->slots * row0);
}

// The records and sums of an evaluation on X; FP64: whatever the mode, the
// FP64 form's only (energy).
int prep_x(pn1_ctx* c, const Phys& P, bool fp64)
{
    MixPrep M = mix_prep(c, P);
    if (fp64) M.j32 = nullptr;
    const bool prev = M.j32 && c->acc_ok;
    // (the energy's sums do not depend on the plan)
    const bool sub = !fp64 && fin_sub(c->n - 1, c->nrow, plan_slots(c));
    hipLaunchKernelGGL(sub ? k_prep<4> : k_prep<1>, dim3((c->nrow + FG - 1) / FG), dim3(FWG), 0,
                       c->st, (const double*)c->X, (const double*)c->m, P, c->nrow, rec_buf(c, 0),
                       row_bufs(c), M, prev ? (const double*)c->acc : nullptr,
                       prev ? (const float*)c->kr : nullptr);
    HIPCHK(c, hipGetLastError());
    return PN1_OK;
}

int enqueue_prep(pn1_ctx* c, const Phys& P) { return prep_x(c, P, false); }

// stage 0: plain evaluation on X; stages 1..3: the driver's force calls.
int enqueue_eval(pn1_ctx* c, int stage, const Phys& P)
{
    const double* in = stage <= 1 ? c->X : c->Y;
    const bool mixed = c->mode == PN1_MIXED;
    const int slots = plan_slots(c);
    if (c->n > 1) {
        hipEvent_t e1 = nullptr;
        if (c->prof) HIPCHK(c, prof_open(c->ev, c->st, &e1));
        const int k = eval_buf(stage);
        if (c->slots)
            launch_pairw(c, k, in, P, 0, c->nrow, stage <= 1);
        else
            launch_pair(c, rec_buf(c, k), in, P, 0, c->nIblk, c->S, stage <= 1);
        if (e1) HIPCHK(c, hipEventRecord(e1, c->st));
    }
    switch (stage * 2 + (mixed ? 1 : 0)) {
    case 0: launch_fin<0, 0>(c, in, P, slots, 1, c->n, true, c->slots > 0); break;
    case 1: launch_fin<1, 0>(c, in, P, slots, 1, c->n, true, c->slots > 0); break;
    case 2: launch_fin<0, 1>(c, in, P, slots, 1, c->n, true, c->slots > 0); break;
    case 3: launch_fin<1, 1>(c, in, P, slots, 1, c->n, true, c->slots > 0); break;
    case 4: launch_fin<0, 2>(c, in, P, slots, 1, c->n, true, c->slots > 0); break;
    case 5: launch_fin<1, 2>(c, in, P, slots, 1, c->n, true, c->slots > 0); break;
    case 6: launch_fin<0, 3>(c, in, P, slots, 1, c->n, true, c->slots > 0); break;
    default: launch_fin<1, 3>(c, in, P, slots, 1, c->n, true, c->slots > 0); break;
    }
    HIPCHK(c, hipGetLastError());
    c->acc_ok = mixed;
    return PN1_OK;
}

// One plain force evaluation of X.
int enqueue_force(pn1_ctx* c, const Phys& P)
{
    const int rc = enqueue_prep(c, P);
    return rc ? rc : enqueue_eval(c, 0, P);
}

int ensure_prev_acc(pn1_ctx* c, const Phys& P)
{
    if (c->mode != PN1_MIXED || c->acc_ok) return PN1_OK;
    const bool prof = c->prof;      // not one of the caller's timed launches
    c->prof = false;
    const int rc = enqueue_force(c, P);
    c->prof = prof;
    return rc;
}

// One step of the driver, its first evaluation prepared (by enqueue_prep or
// the step before).
int enqueue_step(pn1_ctx* c, const Phys& P)
{
    for (int stage = 1; stage <= 3; ++stage) {
        int rc = enqueue_eval(c, stage, P);
        if (rc) return rc;
    }
    return PN1_OK;
}

// ---- between AoS host arrays and SoA device buffers -----------------------
// The finite test adds the exponent's lowest bit to the magnitude's bits,
// which reaches the sign bit for infinities and NaN alone.
static uint64_t copy_finite(const double* a, size_t n, double* out)
{
    uint64_t bad = 0;
    for (size_t k = 0; k < n; ++k) {
        uint64_t b;
        std::memcpy(&b, a + k, sizeof b);
        bad |= (b & 0x7fffffffffffffffull) + 0x0010000000000000ull;
        std::memcpy(out + k, &b, sizeof b);
    }
    return bad >> 63;
}

bool stage_cluster(const double* x, const double* v, const double* m, int n, double* sx,
                   double* sv, double* sm, StarScan* scan)
{
    uint64_t bad = copy_finite(x, 3 * (size_t)n, sx);
    bad |= copy_finite(v, 3 * (size_t)n, sv);
    bad |= copy_finite(m, (size_t)n, sm);
    double mmax = 0.0, dmax2 = 0.0, dmin2 = HUGE_VAL;
    bool differ = false;
    for (int i = 1; i < n; ++i) {
        double d2 = 0.0;
        for (int k = 0; k < 3; ++k) {
            const double d = x[3 * (size_t)i + k] - x[k];
            d2 += d * d;
        }
        dmax2 = d2 > dmax2 ? d2 : dmax2;
        dmin2 = d2 < dmin2 ? d2 : dmin2;
        const double a = std::fabs(m[i]);
        mmax = a > mmax ? a : mmax;
        differ |= m[i] != m[1];
    }
    scan->mmax = mmax;
    scan->dmax2 = dmax2;
    scan->eqm = n < 2 || (!differ && m[1] > 0.0);
    return !bad && m[0] > 0.0 && (n < 2 || dmin2 > 0.0);
}

// Results to the caller's array, large ones 2 KB at a time: their pages are
// often new, and one memcpy faulting them in takes twice as long (3 MB: 660
// us, 330 in pieces; 40 and 45 into pages that are there).
static void copy_out(double* out, const double* stage, size_t n)
{
    const size_t piece = n < (1u << 17) ? n : 256;
    for (size_t k = 0; k < n; k += piece)
        std::memcpy(out + k, stage + k, std::min(piece, n - k) * sizeof(double));
}

// Workgroups of WG threads for cnt values, two each.
static dim3 io_grid(size_t cnt)
{
    return dim3((unsigned)std::max<size_t>(1, (cnt + 2 * WG - 1) / (2 * WG)));
}

int put6(pn1_ctx* c, const double* hx, const double* hv, double* dst, double* zero, size_t nz)
{
    HIPCHK(c, hipStreamSynchronize(c->st));              // the stage is free
    const size_t n3 = 3 * (size_t)c->n;
    if (hx) std::memcpy(c->h_stage, hx, n3 * sizeof(double));
    std::memcpy(c->h_stage + n3, hv, n3 * sizeof(double));
    hipLaunchKernelGGL(k_put, io_grid(std::max(2 * n3, nz)), dim3(WG), 0, c->st, (const double2*)c->h_stage, c->n,
                       (size_t)c->cap, !hx, dst, (double*)nullptr, zero, nz);
    HIPCHK(c, hipGetLastError());
    return PN1_OK;
}

int fetch(pn1_ctx* c, const double* src, int cnt, double* out0, double* out1,
          const double* extra, size_t ne, double* oute)
{
    const size_t n3 = 3 * (size_t)cnt;
    const int nv = out1 ? 2 : 1;
    hipLaunchKernelGGL(k_get, io_grid(nv * n3 + ne), dim3(WG), 0, c->st, src, cnt, (size_t)c->cap,
                       nv, extra, ne, (double2*)c->h_stage);
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipStreamSynchronize(c->st));
    copy_out(out0, c->h_stage, n3);
    if (out1) copy_out(out1, c->h_stage + n3, n3);
    if (ne) std::memcpy(oute, c->h_stage + nv * n3, ne * sizeof(double));
    return PN1_OK;
}

hipError_t copy6(hipStream_t st, double* dst, const double* src, int n, int cap)
{
    hipLaunchKernelGGL(k_copy6, dim3((n + WG - 1) / WG, 6), dim3(WG), 0, st, src, n, (size_t)cap,
                       dst);
    return hipGetLastError();
}

// ---- scratch of pn1_force_noalloc -----------------------------------------
// Sized for n <= PN1_NOALLOC_MAX_N and the explicit_slots of a j split of at
// most NA_MAXS chunks: j-records, pair partials, the rows' values of k_prep and of k_fin_na and its
// counter, each part 256-byte aligned (offsets in doubles).
constexpr int NA_MAXS = 32;
constexpr int NA_MAXB = (PN1_NOALLOC_MAX_N + RB - 1) / RB;
constexpr size_t na_round(size_t d) { return (d + 31) & ~(size_t)31; }
constexpr size_t NA_J64 = 0;
constexpr size_t NA_PART =
    NA_J64 + na_round((size_t)PN1_NOALLOC_MAX_N * (sizeof(JRec64) / sizeof(double)));
constexpr size_t NA_PROWS = NA_PART + na_round((size_t)TLONG * NACC * PN1_NOALLOC_MAX_N);
constexpr size_t NA_ROWV = na_round((size_t)std::max(NA_MAXB, 4 * FIN_SUB) * RV);
constexpr size_t NA_ROWS = NA_PROWS + NA_ROWV;
constexpr size_t NA_TICKET = NA_ROWS + NA_ROWV;
constexpr size_t NA_TOTAL = NA_TICKET + na_round(1);
static_assert(sizeof(JRec64) % sizeof(double) == 0, "JRec64 in doubles");

// j split of pn1_force_noalloc: NA_MAXS chunks, halved while a chunk would
// hold fewer than 64 stars.
int na_split(int nst)
{
    int S = NA_MAXS;
    while (S > 1 && (nst + S - 1) / S < 64) S >>= 1;
    return S;
}

}  // namespace pn1host

using namespace pn1host;

// One per GPU: the code object's __device__ array, placed on each device the
// library runs on when the code object is loaded there, and held until the
// process ends.  Host code never passes its name to a kernel or a copy (on
// the host the name is only a handle): it uses the device address that
// hipGetSymbolAddress returns for the current device (na_scratch).
static __device__ __align__(256) double scratch[NA_TOTAL];

namespace pn1host {

constexpr int NA_MAXDEV = 64;
double* g_na_ptr[NA_MAXDEV];
std::mutex g_na_mu;

// Device address of the current GPU's scratch, looked up once per device.
int na_scratch(int dev, double** out)
{
    std::lock_guard<std::mutex> lock(g_na_mu);
    if (dev < 0 || dev >= NA_MAXDEV) return PN1_ENODEV;
    if (!g_na_ptr[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return PN1_EDEVICE;
        g_na_ptr[dev] = (double*)p;
    }
    *out = g_na_ptr[dev];
    return PN1_OK;
}

}  // namespace pn1host

// =========================================================================
// context API
// =========================================================================
extern "C" {

const char* pn1_last_error(const pn1_ctx* c) { return c ? c->err : "null context"; }

void pn1_destroy(pn1_ctx* c)
{
    if (!c) return;
    if (c->dev >= 0) (void)hipSetDevice(c->dev);
    if (c->st) (void)hipStreamSynchronize(c->st);
    drop_graph(c);
    adj_free(c);
    for (auto& e : c->ev) {
        (void)hipEventDestroy(e.first);
        (void)hipEventDestroy(e.second);
    }
    double* bufs[] = {c->X, c->Y, c->H1, c->H2, c->m, c->acc, c->rows, c->gs, c->eblk};
    for (double* b : bufs)
        if (b) (void)hipFree(b);
    if (c->j64) (void)hipFree(c->j64);
    if (c->j32) (void)hipFree(c->j32);
    if (c->thr) (void)hipFree(c->thr);
    if (c->kr) (void)hipFree(c->kr);
    void* fbufs[] = {c->fmask, c->hmask, c->flist, c->fn, c->ticket, c->xr, c->hpart};
    for (void* b : fbufs)
        if (b) (void)hipFree(b);
    if (c->part) (void)hipFree(c->part);
    if (c->h_stage) (void)hipHostFree(c->h_stage);
    if (c->st) (void)hipStreamDestroy(c->st);
    delete c;
}

int pn1_create(pn1_ctx** out, int capacity, int device)
{
    if (!out) return PN1_EINVAL;
    *out = nullptr;
    if (capacity < 1 || capacity > PN1_MAX_CAPACITY) return PN1_EINVAL;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return PN1_ENODEV;
    if (device < 0 || device >= ndev) return PN1_ENODEV;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) return PN1_ENODEV;
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
        std::fprintf(stderr, "libpn1: device %d is %s; this library is built for gfx950 only\n",
                     device, prop.gcnArchName);
        return PN1_ENODEV;
    }
    pn1_ctx* c = new pn1_ctx;
    c->dev = device;
    c->cap = capacity;
    if (hipSetDevice(device) != hipSuccess ||
        hipStreamCreateWithFlags(&c->st, hipStreamNonBlocking) != hipSuccess) {
        pn1_destroy(c);
        return PN1_EDEVICE;
    }
    const size_t cap = (size_t)capacity;
    const size_t nr = rows_of(cap);                     // rows of 64 stars
    int rc = PN1_OK;
    if (!rc) rc = dalloc(c, &c->X, 6 * cap);
    if (!rc) rc = dalloc(c, &c->Y, 6 * cap);
    if (!rc) rc = dalloc(c, &c->H1, 6 * cap);
    if (!rc) rc = dalloc(c, &c->H2, 6 * cap);
    if (!rc) rc = dalloc(c, &c->m, cap);
    if (!rc) rc = dalloc(c, &c->acc, 3 * cap);
    if (!rc) rc = dalloc(c, &c->rows, std::max(nr, (size_t)4 * FIN_SUB) * RV);
    if (!rc) rc = dalloc(c, &c->gs, 16);
    if (!rc) rc = dalloc(c, &c->eblk, nr * ECHUNK * EV);
    // two records more than particles: the pair loops fetch up to jr[j + 2]
    if (!rc) rc = dalloc(c, &c->j64, 3 * (cap + 2));
    if (!rc) rc = dalloc(c, &c->j32, cap + 2);
    if (!rc) rc = dalloc(c, &c->thr, cap);
    if (!rc) rc = dalloc(c, &c->kr, cap);
    if (!rc) rc = dalloc(c, &c->fmask, nr);
    if (!rc) rc = dalloc(c, &c->hmask, 3 * nr);
    if (!rc) rc = dalloc(c, &c->xr, (size_t)(NACC + 1) * cap);
    if (!rc)
        rc = dalloc(c, &c->hpart,
                    std::min(nr, (size_t)HROWS) * HSLOT * HCHUNK * (NACC + 1));
    if (!rc) rc = dalloc(c, &c->flist, cap);
    if (!rc) rc = dalloc(c, &c->fn, 4);
    if (!rc) rc = dalloc(c, &c->ticket, 1);
    if (!rc && hipMemsetAsync(c->ticket, 0, sizeof(unsigned int), c->st) != hipSuccess)
        rc = PN1_EDEVICE;
    if (!rc && host_malloc((void**)&c->h_stage, stage_doubles(cap, 1) * sizeof(double)) != hipSuccess) {
        c->h_stage = nullptr;
        rc = PN1_ENOMEM;
    }
    if (rc) {
        pn1_destroy(c);
        return rc;
    }
    *out = c;
    return PN1_OK;
}

int pn1_set_params(pn1_ctx* c, double eps, double cl, double dt, int mode)
{
    if (!c) return PN1_EINVAL;
    if (!(eps > 0.0) || !std::isfinite(eps)) return seterr(c, PN1_EINVAL, "eps must be > 0");
    if (!(cl > 0.0) || !std::isfinite(cl)) return seterr(c, PN1_EINVAL, "c must be > 0");
    if (!(dt > 0.0) || !std::isfinite(dt)) return seterr(c, PN1_EINVAL, "dt must be > 0");
    if (mode != PN1_FP64 && mode != PN1_MIXED) return seterr(c, PN1_EINVAL, "unknown mode %d", mode);
    if (eps != c->eps || cl != c->c || dt != c->dt || mode != c->mode) drop_graph(c);
    if (eps != c->eps || cl != c->c || dt != c->dt) ++c->gen;
    // the mixed form's pair thresholds come from the last evaluation's
    // accelerations, which depend on eps and c: take them afresh
    if (eps != c->eps || cl != c->c) c->acc_ok = false;
    c->eps = eps;
    c->c = cl;
    c->dt = dt;
    c->mode = mode;
    return PN1_OK;
}

int pn1_set_tuning(pn1_ctx* c, int jsplit, int tile, int variant)
{
    if (!c) return PN1_EINVAL;
    if (jsplit < 0 || jsplit > 4096 || tile < 0 || tile > 65536 || variant < -1 || variant > 7)
        return seterr(c, PN1_EINVAL, "bad tuning (jsplit %d, tile %d, variant %d)", jsplit, tile,
                      variant);
    const int keep_S = c->jsplit_req, keep_tile = c->tile_req, keep_var = c->variant_req;
    c->jsplit_req = jsplit;
    c->tile_req = tile;
    c->variant_req = variant;
    drop_graph(c);
    if (!c->have_state) return PN1_OK;
    HIPCHK(c, hipSetDevice(c->dev));
    HIPCHK(c, hipStreamSynchronize(c->st));
    const int rc = plan_parts(c);
    if (rc) {                           // refused: the shape in use before stays
        c->jsplit_req = keep_S;
        c->tile_req = keep_tile;
        c->variant_req = keep_var;
        (void)plan_parts(c);
    }
    return rc;
}

int pn1_get_tuning(const pn1_ctx* c, int* jsplit, int* tile, int* variant)
{
    if (!c) return PN1_EINVAL;
    // the row kernels run without a variant alone, the automatic plan's splits
    // of them without a split too
    const bool automatic = c->jsplit_req <= 0 && c->variant_req < 0;
    if (jsplit) *jsplit = automatic ? 0 : c->S;
    if (tile) *tile = c->tile;
    if (variant) *variant = automatic || c->slots ? -1 : kernel_variant(c);
    return PN1_OK;
}

int pn1_upload(pn1_ctx* c, const double* x, const double* v, const double* m, int n)
{
    if (!c) return PN1_EINVAL;
    char msg[256];
    if (n < 1 || !x || !v || !m || n > c->cap) {
        const int rc = pn1_check_input(x, v, m, n, c->eps, msg, sizeof msg);
        if (rc) return seterr(c, rc, "%s", msg);
        return seterr(c, PN1_EINVAL, "n = %d exceeds capacity %d", n, c->cap);
    }
    HIPCHK(c, hipSetDevice(c->dev));
    HIPCHK(c, hipStreamSynchronize(c->st));
    double* h = c->h_stage;
    StarScan scan;
    if (!stage_cluster(x, v, m, n, h, h + 3 * (size_t)n, h + 6 * (size_t)n, &scan)) {
        const int rc = pn1_check_input(x, v, m, n, c->eps, msg, sizeof msg);
        if (rc) return seterr(c, rc, "%s", msg);
    }
    hipLaunchKernelGGL(k_put, io_grid(7 * (size_t)n), dim3(WG), 0, c->st, (const double2*)h, n, (size_t)c->cap,
                       false, c->X, c->m, (double*)nullptr, (size_t)0);
    HIPCHK(c, hipGetLastError());
    // a captured step holds this state's launch constants (n, the BH mass,
    // the mixed form's mass scale, equal-mass kernels, BH-close threshold)
    drop_graph(c);
    ++c->gen;
    c->n = n;
    c->m0 = m[0];
    // mass scale of the mixed records: the largest |m_j| of the stars (0 if
    // every star is massless: their records then have mass 0, and no pair
    // needs a threshold); the equal-mass kernels take unit record masses,
    // so only for stars of one positive mass
    c->mmax = scan.mmax;
    c->eqm = n > 1 && scan.eqm;
    c->tauf = flag_threshold(std::sqrt(scan.dmax2));
    c->acc_ok = false;
    c->have_state = true;
    return plan_parts(c);
}

int pn1_download(pn1_ctx* c, double* x, double* v)
{
    int rc;
    if (!ready(c, &rc)) return rc;
    if (!x || !v) return seterr(c, PN1_EINVAL, "null output");
    return fetch(c, c->X, c->n, x, v);
}

int pn1_force(pn1_ctx* c, double* a)
{
    int rc;
    if (!ready(c, &rc)) return rc;
    if (!a) return seterr(c, PN1_EINVAL, "null output");
    const Phys P = make_phys(c);
    if ((rc = ensure_prev_acc(c, P))) return rc;
    if ((rc = enqueue_force(c, P))) return rc;
    return fetch(c, c->acc, c->n, a, nullptr);
}

int pn1_force_range(pn1_ctx* c, int i0, int i1, double* a)
{
    int rc;
    if (!ready(c, &rc)) return rc;
    if (!a) return seterr(c, PN1_EINVAL, "null output");
    const int n = c->n;
    if (i0 < 1 || i1 > n || i0 >= i1 || (i0 - 1) % WG != 0 || ((i1 - 1) % WG != 0 && i1 != n))
        return seterr(c, PN1_EINVAL,
                      "star range [%d, %d) must lie in [1, %d) and start and end on %d-star "
                      "block boundaries (or end at n)", i0, i1, n, WG);
    const Phys P = make_phys(c);
    const bool mixed = c->mode == PN1_MIXED;
    const double* in = c->X;
    const int nib = (i1 - i0 + WG - 1) / WG;
    // The j split: an explicit one (pn1_set_tuning, pn1_autotune) as set,
    // which keeps the rows bitwise equal to pn1_force's; otherwise the
    // shard's own plan, auto_split doubled while the shard's grid has fewer
    // than 16384 workgroups (chunks of >= 64 records, at most 512 chunks).
    int S = c->jsplit_req > 0 ? c->S : auto_split(n - 1);
    if (c->jsplit_req <= 0) {
        const int nst = n - 1;
        while (S < 512 && (long)S * nib < 16384 && (nst + 2 * S - 1) / (2 * S) >= 64) S *= 2;
    }
    if ((rc = ensure_prev_acc(c, P))) return rc;
    const bool rowk = c->jsplit_req > 0 && c->slots;
    const int slots = rowk ? c->slots : part_slots(c, S);
    if ((rc = ensure_part(c, rowk ? 0 : S))) return rc;
    // every star's j-record and the separable sums: what a sharded run would
    // all-gather and all-reduce before its pair kernel
    if ((rc = enqueue_prep(c, P))) return rc;
    hipEvent_t e1 = nullptr;
    if (c->prof) HIPCHK(c, prof_open(c->ev, c->st, &e1));
    if (rowk)
        launch_pairw(c, 0, in, P, (i0 - 1) / RB, (i1 - i0 + RB - 1) / RB, true);
    else
        launch_pair(c, rec_buf(c, 0), in, P, (i0 - 1) / WG, nib, S, true);
    if (e1) HIPCHK(c, hipEventRecord(e1, c->st));
    if (mixed)
        launch_fin<1, 0>(c, in, P, slots, i0, i1, false, rowk);
    else
        launch_fin<0, 0>(c, in, P, slots, i0, i1, false, rowk);
    if (!mixed) c->acc_ok = false;
    HIPCHK(c, hipGetLastError());
    return fetch(c, c->acc + i0, i1 - i0, a, nullptr);
}

int pn1_energy(pn1_ctx* c, pn1_energy_t* out)
{
    int rc;
    if (!ready(c, &rc)) return rc;
    if (!out) return seterr(c, PN1_EINVAL, "null output");
    const Phys P = make_phys(c);
    if ((rc = prep_x(c, P, true))) return rc;
    hipLaunchKernelGGL(k_energy, dim3(c->nrow, energy_chunks(c->n - 1)), dim3(PW * RB), 0, c->st,
                       (const JRec64*)rec_buf(c, 0), (const double*)c->X, (const double*)c->gs,
                       c->eblk, c->h_stage, c->ticket, P);
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipStreamSynchronize(c->st));
    const double* e = c->h_stage;
    out->kin = e[0];
    out->pot = e[1];
    out->pot_pn = e[2];
    out->pot_pn2 = e[3];
    out->total = e[4];
    return PN1_OK;
}

int pn1_step(pn1_ctx* c, int steps)
{
    int rc;
    if (!ready(c, &rc)) return rc;
    if (steps < 0) return seterr(c, PN1_EINVAL, "steps < 0");
    if (steps == 0) return PN1_OK;
    const Phys P = make_phys(c);
    if ((rc = ensure_prev_acc(c, P))) return rc;
    if ((rc = enqueue_prep(c, P))) return rc;
    if (c->prof) {
        for (int s = 0; s < steps; ++s)
            if ((rc = enqueue_step(c, P))) return rc;
        return PN1_OK;
    }
    if (!c->gexec) {
        hipGraph_t g = nullptr;
        HIPCHK(c, hipStreamBeginCapture(c->st, hipStreamCaptureModeThreadLocal));
        rc = enqueue_step(c, P);
        hipError_t ec = hipStreamEndCapture(c->st, &g);
        if (rc) {
            if (g) (void)hipGraphDestroy(g);
            return rc;
        }
        if (ec != hipSuccess)
            return seterr(c, PN1_EDEVICE, "hipStreamEndCapture failed: %s", hipGetErrorString(ec));
        hipError_t ei = hipGraphInstantiate(&c->gexec, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (ei != hipSuccess) {
            c->gexec = nullptr;
            return seterr(c, PN1_EDEVICE, "hipGraphInstantiate failed: %s", hipGetErrorString(ei));
        }
    }
    for (int s = 0; s < steps; ++s) HIPCHK(c, hipGraphLaunch(c->gexec, c->st));
    return PN1_OK;
}

int pn1_sync(pn1_ctx* c)
{
    if (!c) return PN1_EINVAL;
    HIPCHK(c, hipSetDevice(c->dev));
    HIPCHK(c, hipStreamSynchronize(c->st));
    return PN1_OK;
}

int pn1_profile_enable(pn1_ctx* c, int on)
{
    if (!c) return PN1_EINVAL;
    HIPCHK(c, hipSetDevice(c->dev));
    HIPCHK(c, hipStreamSynchronize(c->st));
    for (auto& e : c->ev) {
        (void)hipEventDestroy(e.first);
        (void)hipEventDestroy(e.second);
    }
    c->ev.clear();
    c->prof = on != 0;
    c->prof_launches = 0;
    c->prof_ms = 0.0;
    return PN1_OK;
}

int pn1_profile_read(pn1_ctx* c, int* launches, double* total_ms)
{
    if (!c) return PN1_EINVAL;
    HIPCHK(c, hipSetDevice(c->dev));
    HIPCHK(c, hipStreamSynchronize(c->st));
    for (auto& e : c->ev) {
        float ms = 0.0f;
        HIPCHK(c, hipEventElapsedTime(&ms, e.first, e.second));
        c->prof_ms += ms;
        c->prof_launches += 1;
        (void)hipEventDestroy(e.first);
        (void)hipEventDestroy(e.second);
    }
    c->ev.clear();
    if (launches) *launches = c->prof_launches;
    if (total_ms) *total_ms = c->prof_ms;
    return PN1_OK;
}

// Autotuner: times the pair kernel of `reps` force evaluations on the
// resident state per candidate shape (j split x kernel variant; the mixed
// form's compensation interval is left alone: it trades accuracy), after
// one warm-up evaluation, and keeps the fastest.  Shapes within TUNE_MARGIN of
// the fastest are timed a second time, each keeping its better one: the first
// shapes run on a clock that is still rising (measured on MI355X, 256 clusters
// of 256-8192 stars, mixed: the automatic plan 2.29 ms first, 2.03 later, the
// next best 2.26).
constexpr double TUNE_MARGIN = 1.25;
int pn1_autotune(pn1_ctx* c, int reps, int* jsplit, int* variant, double* best_ms)
{
    int rc;
    if (!ready(c, &rc)) return rc;
    if (reps < 1) return seterr(c, PN1_EINVAL, "reps must be >= 1");
    const int nst = c->n - 1;
    const bool was_prof = c->prof;
    const int keep_tile = c->tile_req, keep_S = c->jsplit_req, keep_var = c->variant_req;
    std::vector<int> splits = {0};    // 0 = the automatic plan, which has one form
    for (int S = 8; S <= 256; S *= 2)
        if (S <= std::max(1, nst / 64)) splits.push_back(S);
    const Phys P = make_phys(c);
    double best = 1e300;
    int bS = 0, bV = -1;
    // whole force evaluations (every kernel: the partial-sum reduction in
    // k_fin grows with the split), timed with events on the stream
    hipEvent_t ea = nullptr, eb = nullptr;
    if (hipEventCreate(&ea) != hipSuccess || hipEventCreate(&eb) != hipSuccess) {
        if (ea) (void)hipEventDestroy(ea);
        return seterr(c, PN1_EDEVICE, "hipEventCreate failed");
    }
    if ((rc = pn1_profile_enable(c, 0))) {
        (void)hipEventDestroy(ea);
        (void)hipEventDestroy(eb);
        return rc;
    }
    auto time_shape = [&](int S, int var, double* avg) {
        c->jsplit_req = S;
        c->variant_req = S ? var : -1;
        c->tile_req = keep_tile;
        int r = plan_parts(c);
        if (!r) r = enqueue_force(c, P);                         // warm-up
        if (!r && hipEventRecord(ea, c->st) != hipSuccess) r = seterr(c, PN1_EDEVICE, "hipEventRecord failed");
        for (int k = 0; k < reps && !r; ++k) r = enqueue_force(c, P);
        if (!r && hipEventRecord(eb, c->st) != hipSuccess) r = seterr(c, PN1_EDEVICE, "hipEventRecord failed");
        float ms = 0.0f;
        if (!r && (hipEventSynchronize(eb) != hipSuccess || hipEventElapsedTime(&ms, ea, eb) != hipSuccess))
            r = seterr(c, PN1_EDEVICE, "timing the force evaluations failed");
        *avg = (double)ms / reps;
        return r;
    };
    struct Shape {
        int S, var;
        double ms;
    };
    std::vector<Shape> shapes;
    for (int S : splits)
        for (int var = 0; var < (S ? 2 : 1); ++var) shapes.push_back(Shape{S, var, 0.0});
    for (int round = 0; round < 2 && !rc; ++round) {
        const double limit = TUNE_MARGIN * best;
        for (Shape& s : shapes) {
            if (round > 0 && s.ms > limit) continue;
            if ((rc = time_shape(s.S, s.var, &s.ms))) break;
            if (s.ms < best) {
                best = s.ms;
                bS = s.S;
                bV = c->variant_req;
            }
        }
    }
    (void)hipEventDestroy(ea);
    (void)hipEventDestroy(eb);
    (void)pn1_profile_enable(c, was_prof ? 1 : 0);
    if (rc) {                              // leave the shape the caller had
        c->jsplit_req = keep_S;
        c->variant_req = keep_var;
        (void)plan_parts(c);
        return rc;
    }
    c->jsplit_req = bS;
    c->variant_req = bV;
    drop_graph(c);
    if ((rc = plan_parts(c))) return rc;
    if (best_ms) *best_ms = best;
    return pn1_get_tuning(c, jsplit, nullptr, variant);
}

// =========================================================================
// no-allocation force
// =========================================================================
// The FP64 force of pn1_force on a state the caller holds in device memory,
// with every intermediate in this GPU's scratch: the same kernels, the j
// split na_split(n - 1).  Enqueues only (no hipMalloc, hipFree, memset or
// synchronisation); nothing in the scratch needs clearing beforehand, every
// value read is written earlier in the same call, the counter too (a call that
// overlapped another one against the contract leaves nothing behind).  Three
// launches: n = 4097, 103 us with the wait -> 62 (256-star kernels, five
// launches before), n = 257, 45 -> 31.
int pn1_force_noalloc(const double* st, const double* m, int n, double eps, double c,
                      double* acc, void* stream)
{
    if (!st || !m || !acc || n < 1 || n > PN1_NOALLOC_MAX_N) return PN1_EINVAL;
    if (!(eps > 0.0) || !std::isfinite(eps) || !(c > 0.0) || !std::isfinite(c))
        return PN1_EINVAL;
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) return PN1_EDEVICE;
    double* base = nullptr;
    const int rc = na_scratch(dev, &base);
    if (rc) return rc;
    const hipStream_t s = (hipStream_t)stream;
    Phys P;
    P.eps = eps;
    P.eps2 = eps * eps;
    P.lam = 1.0 / (c * c);
    P.dt = 0.0;
    P.m0 = 0.0;                 // the kernels read the BH mass from m[0]
    P.ws = 1.0 / std::sqrt(P.eps2);
    P.mmax = 0.0;
    P.eps2f = (float)P.eps2;
    P.m0f = 0.0f;
    P.n = n;
    P.cap = n;
    JRec64* j64 = (JRec64*)(base + NA_J64);
    double* part = base + NA_PART;
    RowBufs R = {};
    R.rows = base + NA_PROWS;
    R.clear = (unsigned int*)(base + NA_TICKET);
    FinBufs F = {};
    F.in = st;
    F.m = m;
    F.acc = acc;
    F.j64 = j64;
    const int nst = n - 1, nib = (nst + WG - 1) / WG;
    const int nrow = nst > 0 ? (nst + RB - 1) / RB : 1;
    const int S = na_split(nst);
    // (the rows hold fewer than 2^22 / 16 stars here: S = 1 alone is not theirs)
    const int slots = explicit_slots(S, nst);
    const int parts = slots ? slots : S;
    const bool sub = fin_sub(nst, nrow, parts);
    hipLaunchKernelGGL(sub ? k_prep<4> : k_prep<1>, dim3((nrow + FG - 1) / FG), dim3(FWG), 0, s,
                       st, m, P, nrow, j64, R, MixPrep{}, (const double*)nullptr,
                       (const float*)nullptr);
    if (slots)
        hipLaunchKernelGGL(k_pair64w, dim3(slots * nrow), dim3(PW * RB), 0, s, (const JRec64*)j64,
                           st, part, P, slots, nrow, 0);
    else if (nst > 0)
        hipLaunchKernelGGL(k_pair64<0>, dim3(pair_grid(S, nib)), dim3(WG), 0, s,
                           (const JRec64*)j64, st, part, P, S, nib, 0);
    R.rows = base + NA_ROWS;
    R.ticket = (unsigned int*)(base + NA_TICKET);
    hipLaunchKernelGGL(sub ? k_fin_na<4> : k_fin_na<1>, dim3(sub ? 4 * nrow : nrow), dim3(FWG), 0,
                       s, F, R, (const double*)(base + NA_PROWS), (const void*)part, parts, P,
                       nrow);
    return hipGetLastError() == hipSuccess ? PN1_OK : PN1_EDEVICE;
}

// =========================================================================
// legacy shapes
// =========================================================================
static pn1_ctx* g_ctx = nullptr;
static double g_c = 1.0;
static int g_mode = PN1_FP64;

int pn1_set_c(double cl)
{
    if (!(cl > 0.0) || !std::isfinite(cl)) return PN1_EINVAL;
    g_c = cl;
    return PN1_OK;
}

int pn1_set_mode(int mode)
{
    if (mode != PN1_FP64 && mode != PN1_MIXED) return PN1_EINVAL;
    g_mode = mode;
    return PN1_OK;
}

static void die(const char* what, const char* msg)
{
    std::fprintf(stderr, "%s: %s\n", what, msg);
    std::exit(1);
}

static pn1_ctx* legacy_ctx(const char* what, const double* x, const double* v, const double* m,
                           int n, double eps, int mode)
{
    char msg[256];
    if (!g_ctx || g_ctx->cap < n) {
        if (pn1_check_input(x, v, m, n, eps, msg, sizeof msg) != PN1_OK) die(what, msg);
        pn1_destroy(g_ctx);
        g_ctx = nullptr;
        int cap = n < 1024 ? 1024 : n;
        int rc = pn1_create(&g_ctx, cap, 0);
        if (rc != PN1_OK) {
            std::snprintf(msg, sizeof msg, "cannot create a gfx950 device context (status %d)", rc);
            die(what, msg);
        }
    }
    if (pn1_set_params(g_ctx, eps, g_c, g_ctx->dt, mode) != PN1_OK ||
        pn1_upload(g_ctx, x, v, m, n) != PN1_OK) {
        if (pn1_check_input(x, v, m, n, eps, msg, sizeof msg) != PN1_OK) die(what, msg);
        die(what, g_ctx->err);
    }
    return g_ctx;
}

void force(double (*x)[3], double (*v)[3], double* m, double eps, double (*a)[3], double* pot, int n)
{
    (void)pot;  // ignored, as in Limit-sticky9.c:21-424
    pn1_ctx* c = legacy_ctx("force", &x[0][0], &v[0][0], m, n, eps, g_mode);
    if (pn1_force(c, &a[0][0]) != PN1_OK) die("force", c->err);
}

static void legacy_energy(const char* what, double (*x)[3], double (*v)[3], double* m, int n,
                          double eps, pn1_energy_t* e)
{
    pn1_ctx* c = legacy_ctx(what, &x[0][0], &v[0][0], m, n, eps, PN1_FP64);
    if (pn1_energy(c, e) != PN1_OK) die(what, c->err);
}

// The print block of Limit-sticky9.c:560-563 / 701-703.
static void print_block(double t, const pn1_energy_t* e)
{
    std::printf("time = %g\n", t);
    std::printf("pot = %22.15e kin = %22.15e \n pot_pn = %22.15e \n  total= %22.15e ratio = %e\n",
                e->pot, e->kin, e->pot_pn, e->total, e->kin / e->pot);
}

void energy(double t, double (*x)[3], double (*v)[3], double* m, int n, double init_ene, double eps)
{
    pn1_energy_t e;
    legacy_energy("energy", x, v, m, n, eps, &e);
    const double de = (init_ene - e.total) / e.total;
    print_block(t, &e);
    std::printf(" DE = %e %g\n", de, t);
}

void initial_energy(double (*x)[3], double (*v)[3], double* m, int n, double* init_ene, double eps)
{
    pn1_energy_t e;
    legacy_energy("initial_energy", x, v, m, n, eps, &e);
    print_block(0.0, &e);
    *init_ene = e.total;
}

}  // extern "C"

#include "pn1_ens.inc"
