// CPU check of the ensemble's automatic chunk (pn_amd/csrc/pn1_ens_plan.hpp):
// for each line "clusters stars" (clusters of that many stars each) on stdin,
// prints the chunk and the workgroups it gives.  Run by
// tests/test_ens_plan_host.py.
#include <cstdio>

#include "pn1_ens_plan.hpp"

int main()
{
    long nc, ns;
    while (std::scanf("%ld %ld", &nc, &ns) == 2) {
        std::vector<int> off(nc + 1);
        for (long c = 0; c <= nc; ++c) off[c] = (int)(c * (ns + 1));
        const int L = pn1host::ens_auto_chunk(off);
        std::printf("%ld %ld %d %ld\n", nc, ns, L, L > 0 ? pn1host::ens_parts(off, L) : -1);
    }
    return 0;
}
