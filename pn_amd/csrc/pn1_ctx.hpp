// pn1_ctx.hpp -- the context behind pn1_ctx* (private to libpn1), shared by
// the translation units of the library: pn1_api.hip (force, energy, stage
// driver, legacy shapes, ensembles) and pn1_adj.hip (adjoint).
#pragma once
#include <hip/hip_runtime.h>

#include <utility>
#include <vector>

#include "pn1.h"
#include "pn1_common.hpp"

struct pn1_adj;   // adjoint buffers (pn1_adj.hip)

struct pn1_ctx {
    int dev = -1;
    hipStream_t st = nullptr;
    int cap = 0, n = 0;
    bool have_state = false;
    double eps = 1e-3, c = 1.0, dt = 1.0 / 1024.0;
    int mode = PN1_FP64;
    double m0 = 0.0;            // host copy of m[0]
    double mmax = 0.0;          // largest star mass (mixed form's pair thresholds)
    bool eqm = false;           // every star has the same mass
    double tauf = 0.0;          // BH-close threshold of the mixed form (PN1_FLAG_ETA)
    int jsplit_req = 0, tile_req = 0, variant_req = -1;
    // launch plan for the current n
    // j split (S parts); slots: partials per star of the automatic plan's pair
    // kernels, which give each PW parts (0: the explicit split's kernels)
    int S = 1, slots = 0, nIblk = 0, tile = 64;
    // device buffers
    double *X = nullptr, *Y = nullptr, *H1 = nullptr, *H2 = nullptr;
    double *m = nullptr, *acc = nullptr, *rows = nullptr, *gs = nullptr;
    double* eblk = nullptr;
    // three buffers of cap + 2 records: each of a step's evaluations reads
    // one and prepares the next
    pn1dev::JRec64* j64 = nullptr;
    pn1dev::JRec32* j32 = nullptr;
    pn1dev::Thr* thr = nullptr; // mixed form's per-star pair thresholds
    float* kr = nullptr;        // mixed form's per-star cancellation ratios
    // per row of 64 stars: its values of the sums over all stars (rows) and,
    // mixed form, the masks of its BH-close and hard stars (hmask: three of
    // rows_of(cap), one to each record buffer); the list of BH-close stars and
    // its length; the O(n) kernels' ticket counter
    int nrow = 1;
    unsigned long long *fmask = nullptr, *hmask = nullptr;
    int *flist = nullptr, *fn = nullptr;
    unsigned int* ticket = nullptr;
    double* xr = nullptr;       // FP64 sums for hard stars and BH-close pairs [NACC + 1][cap]
    double* hpart = nullptr;    // hard stars' sums of the row kernels, [rows][HSLOT][HCHUNK][NACC + 1]
    // acc and kr hold the last mixed evaluation of the uploaded run (cleared
    // by pn1_upload and by FP64 evaluations): the mixed form's thresholds
    // read them
    bool acc_ok = false;
    void* part = nullptr;
    size_t part_bytes = 0;
    double* h_stage = nullptr;  // pinned, stage_doubles(cap, 1)
    hipGraphExec_t gexec = nullptr;
    bool prof = false;
    std::vector<std::pair<hipEvent_t, hipEvent_t>> ev;
    int prof_launches = 0;
    double prof_ms = 0.0;
    pn1_adj* adj = nullptr;     // allocated by the first adjoint call
    unsigned gen = 0;           // bumped when the state, masses or parameters change
    char err[512] = {0};
};

namespace pn1host {

int seterr(pn1_ctx* c, int code, const char* fmt, ...);
pn1dev::Phys make_phys(const pn1_ctx* c);
// The records and sums of a plain evaluation or a step's first one, on X.
int enqueue_prep(pn1_ctx* c, const pn1dev::Phys& P);
// One prepared evaluation on the context's stream (stage 0: plain, on X;
// 1..3: the stage driver's calls, with their state updates, each preparing
// the next; stage 3 the next step's first).
int enqueue_eval(pn1_ctx* c, int stage, const pn1dev::Phys& P);
// Mixed form after an upload: one evaluation with the pair thresholds off
// (no previous accelerations yet), so that the next has them.
int ensure_prev_acc(pn1_ctx* c, const pn1dev::Phys& P);
// ---- between AoS host arrays and SoA device buffers (pn1_io.hpp)
// Doubles of the stage of a context or ensemble: a state, and per cluster
// what is fetched with it (gm0) or instead of it (the energies).
// (an even number: the kernels take double2)
inline size_t stage_doubles(size_t cap, size_t clusters)
{
    return (7 * cap + 8 * clusters + 1) / 2 * 2;
}
// What the launches need of a cluster's stars: the largest |m|, the largest
// squared distance to the BH, whether all have one positive mass.
struct StarScan {
    double mmax = 0.0, dmax2 = 0.0;
    bool eqm = true;
};
// Copies a cluster (BH first) to sx, sv, sm and scans its stars.  False if
// pn1_check_input might refuse it (it then says).
bool stage_cluster(const double* x, const double* v, const double* m, int n, double* sx,
                   double* sv, double* sm, StarScan* scan);
// The caller's arrays hx (null: zeros) and hv into the stage and on to dst (6
// x cap); clears zero[0, nz).
int put6(pn1_ctx* c, const double* hx, const double* hv, double* dst, double* zero, size_t nz);
// src (SoA, cnt stars from its first) to out0 and, if not null, src + 3 cap to
// out1, AoS; also extra[0, ne) to oute.  Waits for the stream.
int fetch(pn1_ctx* c, const double* src, int cnt, double* out0, double* out1,
          const double* extra = nullptr, size_t ne = 0, double* oute = nullptr);
hipError_t copy6(hipStream_t st, double* dst, const double* src, int n, int cap);
// Checks that a state is resident and makes the context's device current;
// *rc is PN1_OK, or the error when it returns false.
bool ready(pn1_ctx* c, int* rc);
void drop_graph(pn1_ctx* c);
void adj_free(pn1_ctx* c);   // pn1_adj.hip

}  // namespace pn1host

// hipMalloc / hipHostMalloc whose failure is returned as a status only: HIP
// also keeps a failed call's code for the next hipGetLastError(), which the
// launch checks read, so a refused allocation would otherwise fail the next,
// valid launch.  *p is null on failure.
inline hipError_t dev_malloc(void** p, size_t bytes)
{
    const hipError_t r = hipMalloc(p, bytes);
    if (r != hipSuccess) {
        *p = nullptr;
        (void)hipGetLastError();
    }
    return r;
}

inline hipError_t host_malloc(void** p, size_t bytes)
{
    const hipError_t r = hipHostMalloc(p, bytes);
    if (r != hipSuccess) {
        *p = nullptr;
        (void)hipGetLastError();
    }
    return r;
}

// Opens a timed region on stream `st`: two events handed to `ev` at once
// (so a later error leaks neither), the first recorded now; the caller
// records *end after the launches it times.
inline hipError_t prof_open(std::vector<std::pair<hipEvent_t, hipEvent_t>>& ev, hipStream_t st,
                            hipEvent_t* end)
{
    hipEvent_t a = nullptr, b = nullptr;
    hipError_t r = hipEventCreate(&a);
    if (r != hipSuccess) return r;
    if ((r = hipEventCreate(&b)) != hipSuccess) {
        (void)hipEventDestroy(a);
        return r;
    }
    ev.emplace_back(a, b);
    *end = b;
    return hipEventRecord(a, st);
}

#define HIPCHK(ctx, call)                                                                 \
    do {                                                                                  \
        hipError_t e_ = (call);                                                           \
        if (e_ != hipSuccess)                                                             \
            return seterr((ctx), PN1_EDEVICE, "%s failed: %s", #call, hipGetErrorString(e_)); \
    } while (0)

