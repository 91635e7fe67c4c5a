// pn1_ens.hpp -- the ensemble behind pn1_ens* (private to libpn1), shared by
// pn1_api.hip (force, energy, steps: pn1_ens.inc) and pn1_adj.hip (adjoint).
//
// Device layout: one state of capacity cap (SoA, as pn1_ctx) holding all
// clusters back to back; per cluster its BH first.  Tables built at upload:
//   coff[nc + 1]   first particle of each cluster
//   cm0[nc]        BH mass of each cluster
//   cmmax[nc]      largest star mass of each cluster
//   row[nrow], crow[nc + 1]   64-star rows of the O(n) kernels, per
//                  cluster; pblk[npblk]: groups of FG of them
//   parts[nparts]  the automatic plan's pair work items (row, chunk), filled
//                  on the device from place[nc]
//   items[nitems]  the 256-star items of an explicit chunk or variant and of
//                  the adjoint, in 8 per-XCD queues (qoff[9]): whole
//                  clusters go to the least-loaded queue, largest first;
//                  each queue is sorted by decreasing pair count; built when
//                  first needed
//   poff[nc]       first partial-sum slot of each cluster
#pragma once
#include <hip/hip_runtime.h>

#include <utility>
#include <vector>

#include "pn1.h"
#include "pn1_ens_plan.hpp"
#include "pn1_ens_types.hpp"

struct pn1_ens_adj;   // adjoint buffers (pn1_adj.hip)

struct pn1_ens {
    int dev = -1;
    hipStream_t st = nullptr;
    int cap = 0, capc = 0, n = 0, nc = 0;
    bool have_state = false;
    double eps = 1e-3, c = 1.0, dt = 1.0 / 1024.0;
    int mode = PN1_FP64;
    int L_req = 0, tile_req = 0, variant_req = -1;
    int L = 512, tile = 64;
    double *X = nullptr, *Y = nullptr, *H1 = nullptr, *H2 = nullptr, *m = nullptr, *acc = nullptr;
    double *rows = nullptr, *gs = nullptr, *eblk = nullptr;
    // the tables of the upload, one device block (tab) and its pinned source
    // (h_tab): cm0 ... place below point into it
    char *tab = nullptr, *h_tab = nullptr;
    size_t tab_bytes = 0;
    double* cm0 = nullptr;
    double* cmmax = nullptr;      // each cluster's largest star mass
    pn1dev::Thr* thr = nullptr;   // mixed form's per-star pair thresholds
    float* kr = nullptr;          // mixed form's per-star cancellation ratios
    bool acc_ok = false;          // acc, kr hold the last mixed evaluation
    bool eqm = false;             // each cluster's stars have one mass
    double* ctauf = nullptr;      // each cluster's BH-close threshold (PN1_FLAG_ETA)
    // per row: its values of the sums over all stars (rows) and, mixed form,
    // the masks of its BH-close and hard stars (hmask: three of nrow, one to
    // each record buffer); BH-close stars (lists at each
    // cluster's offset, per-cluster numbers); the O(n) kernels' tickets
    unsigned long long *fmask = nullptr, *hmask = nullptr;
    int *flist = nullptr, *fn = nullptr;
    unsigned int* ticket = nullptr;
    double* xr = nullptr;         // as in pn1_ctx
    double* hpart = nullptr;      // as in pn1_ctx, by the ensemble's rows
    size_t hpart_cap = 0;
    pn1dev::EBlk *row = nullptr, *pblk = nullptr;
    int* crow = nullptr;
    int nrow = 0, npblk = 0;
    size_t fmask_cap = 0, hmask_cap = 0, rows_cap = 0, eblk_cap = 0;
    // three buffers of cap + 2 records, as in pn1_ctx
    pn1dev::JRec64* j64 = nullptr;
    pn1dev::JRec32* j32 = nullptr;
    int *coff = nullptr, *qoff = nullptr;
    pn1dev::EItem* items = nullptr;
    long long* poff = nullptr;
    unsigned int* counter = nullptr;
    int nitems = 0;
    size_t items_cap = 0;
    bool have_items = false;      // items, qoff are those of this state and L
    pn1dev::EPart* parts = nullptr;
    pn1dev::EPlace* place = nullptr;
    int nparts = 0;
    size_t parts_cap = 0;
    bool autoplan = true;         // no explicit chunk at the last upload
    int L_auto = 0;               // the automatic plan's chunk; 0: it does not take this state
    bool tab_auto = false;        // the tables are the automatic plan's
    int Lf = 512;                 // the force's chunk: L or L_auto
    int echunks = 1;                // largest energy_chunks of a cluster
    long long slots = 0;
    void* part = nullptr;
    size_t part_bytes = 0;
    double* h_stage = nullptr;    // pinned, stage_doubles(cap, capc)
    int grid64[2] = {0, 0}, grid32[4] = {0, 0, 0, 0};   // per kernel variant
    hipGraphExec_t gexec = nullptr;
    bool prof = false;
    std::vector<std::pair<hipEvent_t, hipEvent_t>> ev;
    int prof_launches = 0;
    double prof_ms = 0.0;
    pn1_ens_adj* adj = nullptr;   // allocated by the first adjoint call
    unsigned gen = 0;             // bumped when the state or eps, c, dt change
    std::vector<int> off_h;       // host copies: cluster offsets, and per cluster
    std::vector<double> m0_h, mmax_h, tauf_h;   // the values of cm0, cmmax, ctauf
    char err[512] = {0};
};

namespace pn1host {

int eerr(pn1_ens* e, int code, const char* fmt, ...);
pn1dev::Phys ens_phys(const pn1_ens* e);
// Grid of n workgroups whose index is ens_block.
dim3 ens_grid(int n);
// As enqueue_prep and enqueue_eval, for every cluster.
int ens_enqueue_prep(pn1_ens* e, const pn1dev::Phys& P);
int ens_enqueue_eval(pn1_ens* e, int stage, const pn1dev::Phys& P);
// Mixed form after an upload: one evaluation with the pair thresholds off.
int ens_ensure_prev_acc(pn1_ens* e, const pn1dev::Phys& P);
// As put6 and fetch (pn1_ctx.hpp), all particles.
int ens_put6(pn1_ens* e, const double* hx, const double* hv, double* dst, double* zero,
             size_t nz);
int ens_fetch(pn1_ens* e, const double* src, double* out0, double* out1,
              const double* extra = nullptr, size_t ne = 0, double* oute = nullptr);
bool ens_ready(pn1_ens* e, int* rc);
// ens_ready, and the tables are those of the force's present plan.
bool ens_force_ready(pn1_ens* e, int* rc);
// items and qoff for the present state and L, if they are not there.
int ens_items(pn1_ens* e);
void edrop_graph(pn1_ens* e);
void ens_adj_free(pn1_ens* e);   // pn1_adj.hip

}  // namespace pn1host

#define EHIPCHK(e, call)                                                                  \
    do {                                                                                  \
        hipError_t e_ = (call);                                                           \
        if (e_ != hipSuccess)                                                             \
            return eerr((e), PN1_EDEVICE, "%s failed: %s", #call, hipGetErrorString(e_)); \
    } while (0)
