// CPU check of what an ensemble launches after refused allocations, over the
// runtime of fake_hip.hpp: each allocation of a plan change, an upload and the
// tuner is refused in turn.  Run by tests/test_fake_hip_host.py; prints
// "ok <cases>".
#include "fake_hip.hpp"
#include "pn1.h"

namespace {

struct State {
    std::vector<int> off;
    std::vector<double> x, v, m;
    explicit State(const std::vector<int>& stars) : off(1, 0)
    {
        for (int s : stars) off.push_back(off.back() + s + 1);
        const int n = off.back();
        for (int i = 0; i < n; ++i) {
            for (int k = 0; k < 3; ++k) {
                x.push_back(0.001 * ((i * 7919 + k * 104729) % 9973) + i);
                v.push_back(0.0);
            }
            m.push_back(1.0 + i % 3);
        }
    }
    int n() const { return off.back(); }
    int upload(pn1_ens* e) const
    {
        particles = n();
        return pn1_ens_upload(e, (int)off.size() - 1, off.data(), x.data(), v.data(), m.data());
    }
};

}  // namespace

int main()
{
    const State one({300}), many(std::vector<int>(400, 1)), mid({600, 5, 0, 64, 2000});
    std::vector<double> a(3 * 4000), en(5 * 400);
    int cases = 0;
    // A plan change after the upload, with each of its allocations refused in
    // turn: the call fails, so does the next one if its own is refused, the
    // energies (which need no plan) go on, and without a refusal all is well.
    for (int mode : {PN1_FP64, PN1_MIXED})
        for (const State* s : {&many, &mid})
            for (int to_items = 0; to_items < 2; ++to_items) {
                const std::string label = "mode " + std::to_string(mode) + ", " +
                                          std::to_string(s->n()) + " particles, to " +
                                          (to_items ? "items" : "the automatic plan");
                for (long k = 0;; ++k) {
                    pn1_ens* e = nullptr;
                    want(pn1_ens_create(&e, 4000, 400, 0), PN1_OK, "create");
                    want(pn1_ens_set_params(e, 1e-2, 10.0, 1e-3, mode), PN1_OK, "params");
                    // items (few) of an earlier state, and the plan to leave
                    want(pn1_ens_set_tuning(e, 0, 0, 0), PN1_OK, "tuning");
                    want(one.upload(e), PN1_OK, "first upload");
                    want(pn1_ens_force(e, a.data()), PN1_OK, "first force");
                    want(pn1_ens_set_tuning(e, 0, 0, to_items ? -1 : 0), PN1_OK, "tuning");
                    want(s->upload(e), PN1_OK, "upload");
                    want(pn1_ens_force(e, a.data()), PN1_OK, "force");
                    want(pn1_ens_set_tuning(e, 0, 0, to_items ? 0 : -1), PN1_OK, "tuning");
                    refuse = k;
                    const int rc = pn1_ens_force(e, a.data());
                    const bool refused = refuse < 0;
                    refuse = -1;
                    if (!refused && k == 0) fail(label + ": nothing to refuse");
                    want(rc, refused ? PN1_ENOMEM : PN1_OK, label + ", change");
                    launched.clear();
                    want(pn1_ens_energy(e, en.data()), PN1_OK, label + ", energy");
                    if (refused) {
                        refuse = 0;                     // the first one it makes
                        want(pn1_ens_force(e, a.data()), PN1_ENOMEM, label + ", again");
                        if (ran("k_ens_pair")) fail(label + ": launched after a refusal");
                        refuse = -1;
                    }
                    launched.clear();
                    want(pn1_ens_force(e, a.data()), PN1_OK, label + ", at last");
                    if (!ran(to_items ? (mode == PN1_MIXED ? "k_ens_pair32<" : "k_ens_pair64<")
                                      : (mode == PN1_MIXED ? "k_ens_pair32w<" : "k_ens_pair64w(")))
                        fail(label + ": wrong kernel");
                    want(pn1_ens_force_vjp(e, a.data(), a.data(), a.data(), nullptr), PN1_OK,
                         label + ", vjp");
                    pn1_ens_destroy(e);
                    ++cases;
                    if (!refused) break;
                }
            }
    // An upload with each allocation refused: withdrawn, and the next one works.
    for (int variant : {-1, 0})
        for (long k = 0;; ++k) {
            pn1_ens* e = nullptr;
            want(pn1_ens_create(&e, 4000, 400, 0), PN1_OK, "create");
            want(pn1_ens_set_tuning(e, 0, 0, variant), PN1_OK, "tuning");
            want(one.upload(e), PN1_OK, "first upload");
            refuse = k;
            const int rc = mid.upload(e);
            const bool refused = refuse < 0;
            refuse = -1;
            want(rc, refused ? PN1_ENOMEM : PN1_OK, "upload");
            want(pn1_ens_energy(e, en.data()), refused ? PN1_EINVAL : PN1_OK, "energy after it");
            want(pn1_ens_force(e, a.data()), refused ? PN1_EINVAL : PN1_OK, "force after it");
            want(many.upload(e), PN1_OK, "next upload");
            want(pn1_ens_force(e, a.data()), PN1_OK, "its force");
            pn1_ens_destroy(e);
            ++cases;
            if (!refused) break;
        }
    // The tuner with each allocation refused: the shape before it, or no state.
    for (long k = 0;; ++k) {
        pn1_ens* e = nullptr;
        want(pn1_ens_create(&e, 4000, 400, 0), PN1_OK, "create");
        want(mid.upload(e), PN1_OK, "upload");
        refuse = k;
        const int rc = pn1_ens_autotune(e, 1, nullptr, nullptr, nullptr);
        const bool refused = refuse < 0;
        refuse = -1;
        want(rc, refused ? PN1_ENOMEM : PN1_OK, "autotune");
        want(pn1_ens_force(e, a.data()), PN1_OK, "force after it");
        pn1_ens_destroy(e);
        ++cases;
        if (!refused) break;
    }
    for (auto& b : blocks)
        if (b.second.live) fail("a block is still allocated");
    std::printf("ok %d\n", cases);
    return 0;
}
