// CPU check of the tuners' choice, over the runtime of fake_hip.hpp: the first
// shape timed runs on a cold clock (an eighth slower), and is the fastest all
// the same.  Run by tests/test_fake_hip_host.py; prints "ok".
#include "fake_hip.hpp"
#include "pn1.h"

namespace {

const char* fast = "";          // the kernel of the fastest shape
int timed = 0;

float by_kernel()
{
    const float warm = ran(fast) ? 3.57f : 3.75f;
    launched.clear();
    return timed++ == 0 ? 1.13f * warm : warm;
}

}  // namespace

int main()
{
    elapsed = by_kernel;
    std::vector<double> x, v(3 * 3001, 0.0), m(3001, 1.0);
    for (int i = 0; i < 3 * 3001; ++i) x.push_back(i % 3 ? i * 0.25 : i * 0.5);
    for (int mode : {PN1_FP64, PN1_MIXED}) {
        int S = 0, var = 0;
        double ms = 0.0;
        pn1_ctx* c = nullptr;
        fast = mode == PN1_MIXED ? "k_pair32w<" : "k_pair64w(";
        timed = 0;
        want(pn1_create(&c, 3001, 0), PN1_OK, "create");
        want(pn1_set_params(c, 1e-2, 10.0, 1e-3, mode), PN1_OK, "params");
        want(pn1_upload(c, x.data(), v.data(), m.data(), 3001), PN1_OK, "upload");
        want(pn1_autotune(c, 1, &S, &var, &ms), PN1_OK, "autotune");
        if (S != 0 || var != -1 || ms > 3.6) fail("context: split " + std::to_string(S));
        pn1_destroy(c);
        pn1_ens* e = nullptr;
        fast = mode == PN1_MIXED ? "k_ens_pair32w<" : "k_ens_pair64w(";
        timed = 0;
        const int off[] = {0, 1001, 3001};
        particles = 3001;
        want(pn1_ens_create(&e, 3001, 2, 0), PN1_OK, "create");
        want(pn1_ens_set_params(e, 1e-2, 10.0, 1e-3, mode), PN1_OK, "params");
        want(pn1_ens_upload(e, 2, off, x.data(), v.data(), m.data()), PN1_OK, "upload");
        want(pn1_ens_autotune(e, 1, &S, &var, &ms), PN1_OK, "autotune");
        if (var != -1 || ms > 3.6) fail("ensemble: chunk " + std::to_string(S));
        pn1_ens_destroy(e);
    }
    std::printf("ok\n");
    return 0;
}
