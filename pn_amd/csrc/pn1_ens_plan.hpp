// pn1_ens_plan.hpp -- sizes of an ensemble's launches, from its clusters'
// offsets alone (plain C++, also compiled by the host tests).
#pragma once
#include <algorithm>
#include <vector>

namespace pn1host {

inline int nchunks_host(int nst, int L) { return (int)(((long)nst + L - 1) / L); }

// Workgroups (rows of 64 stars x chunks of L) of the automatic plan.
inline long ens_parts(const std::vector<int>& off, int L)
{
    long t = 0;
    for (size_t c = 0; c + 1 < off.size(); ++c) {
        const long nst = off[c + 1] - off[c] - 1;
        t += (nst + 63) / 64 * nchunks_host((int)nst, L);
    }
    return t;
}

// Most workgroups of that plan (a launch holds less than 2^32 threads, a
// workgroup 512).
constexpr long ENS_PARTS_MAX = 1L << 22;

// The automatic plan's chunk, of 64 x L pairs per workgroup.  Long chunks pay
// a workgroup's start and end, and the partials in k_ens_fin, less often;
// short ones fill the chip (1024 workgroups are resident) and leave less to
// wait for at the end: 4096, halved down to 512 while there are fewer than
// 6000 workgroups, further, to a wave's 8 records, while fewer than 1024.
// Measured on MI355X (one evaluation, mixed / FP64, us; the rule's in brackets):
//   clusters of        L = 64     128        512        1024       4096
//   256: 256-8192      5430/7530  3840/6020  2670/4720  2500/4630 [2360/4360]
//   12: 4000-9000      823/1150   591/939              [437/737]   522/897
//   100: 400-4000      781/1039   561/831              [420/651]   397/632
//   40: 64-1500        40.8/38.8 [37.5/35.6] 45.4/43.7  58/61      77/59
//   8: 32-600         [25.6/18.6] 27.9/20.3  47.1/34.9  51.7/43.4  51.7/43.4
// (the 256-star items at their L: 256 clusters 2690, 4680)
// Doubled while there are more than ENS_PARTS_MAX; 0 if there still are with
// one chunk per cluster (over 2^22 rows, as of so many small clusters): the
// 256-star items, whose launch is as large as the chip, then take the force.
inline int ens_auto_chunk(const std::vector<int>& off)
{
    int most = 0;
    for (size_t c = 0; c + 1 < off.size(); ++c) most = std::max(most, off[c + 1] - off[c] - 1);
    int L = 4096;
    while (L > 512 && ens_parts(off, L) < 6000) L /= 2;
    while (L > 64 && ens_parts(off, L) < 1024) L /= 2;
    while (ens_parts(off, L) > ENS_PARTS_MAX) {
        if (L >= most) return 0;
        L *= 2;
    }
    return L;
}

}  // namespace pn1host
