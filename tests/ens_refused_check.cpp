// CPU check of what an ensemble launches after refused allocations.
//
// Defines the HIP runtime's entry points that libpn1.so calls, over host
// memory: allocations are registered (and only marked dead when freed), one of
// them can be refused, and a launch, which runs nothing, has its arguments
// checked instead: every pointer (also those of EnsBufs) must lie in a live
// allocation, and the work items a pair kernel gets must be the state's.  The
// executable exports them, so the library's calls end here.  Run by
// tests/test_ens_refused_host.py; prints "ok <cases>".
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "pn1.h"

namespace {

struct Block {
    size_t bytes;
    bool live;
};
std::map<const char*, Block> blocks;
// host stub -> demangled kernel (the library registers them as it is loaded,
// before this file's own objects exist)
std::map<const void*, std::string>& names()
{
    static std::map<const void*, std::string> m;
    return m;
}
long refuse = -1;                              // allocations until one is refused
std::vector<std::string> launched;
int particles = 0;                             // of the state uploaded
dim3 cfg_g, cfg_b;
size_t cfg_sh;
hipStream_t cfg_s;

[[noreturn]] void fail(const std::string& what)
{
    std::printf("FAILED %s\n", what.c_str());
    std::exit(1);
}

// Bytes from p to the end of its live block (0: none).
size_t room(const void* p)
{
    auto it = blocks.upper_bound((const char*)p);
    if (it == blocks.begin()) return 0;
    --it;
    const size_t at = (size_t)((const char*)p - it->first);
    return it->second.live && at < it->second.bytes ? it->second.bytes - at : 0;
}

hipError_t give(void** p, size_t n)
{
    if (refuse == 0) {
        refuse = -1;
        *p = nullptr;
        return hipErrorOutOfMemory;
    }
    if (refuse > 0) --refuse;
    *p = std::calloc(n, 1);
    blocks[(const char*)*p] = Block{n, true};
    return hipSuccess;
}

hipError_t take(void* p)
{
    if (!p) return hipSuccess;
    auto it = blocks.find((const char*)p);
    if (it == blocks.end() || !it->second.live) fail("free of an unknown block");
    it->second.live = false;
    return hipSuccess;
}

// The parameter types of a demangled kernel.
std::vector<std::string> params(const std::string& sig)
{
    size_t open = sig.find('(');
    int depth = 0;
    for (size_t i = 0; i < sig.size(); ++i) {
        if (sig[i] == '<') ++depth;
        if (sig[i] == '>') --depth;
        if (sig[i] == '(' && depth == 0) {
            open = i;
            break;
        }
    }
    std::vector<std::string> out;
    std::string cur;
    for (size_t i = open + 1; i < sig.size(); ++i) {
        if (sig[i] == '<') ++depth;
        if (sig[i] == '>') --depth;
        if (depth == 0 && (sig[i] == ',' || sig[i] == ')')) {
            out.push_back(cur);
            cur.clear();
            if (sig[i] == ')') break;
        } else {
            cur += sig[i];
        }
    }
    return out;
}

// As EItem (pn1_ens_types.hpp).
struct Item {
    int off, nst, ib, j0, j1, c;
    long long pslot;
};

void check(const std::string& sig, void** args)
{
    const std::vector<std::string> ps = params(sig);
    const int* qoff = nullptr;
    const Item* items = nullptr;
    size_t part = 0;
    auto ptr = [&](size_t k) {
        void* p;
        std::memcpy(&p, args[k], sizeof p);
        return (const void*)p;
    };
    for (size_t k = 0; k < ps.size(); ++k) {
        if (ps[k].find('*') != std::string::npos) {
            const void* p = ptr(k);
            if (p && !room(p)) fail(sig + ": argument " + std::to_string(k) + " is not live");
            if (ps[k].find("EItem") != std::string::npos) {
                items = (const Item*)p;
                qoff = (const int*)ptr(k + 2);          // items, counter, qoff
                // (the adjoint's are laid out otherwise)
                part = sig.find("k_ens_pair") != std::string::npos ? room(ptr(k - 1)) : SIZE_MAX;
            }
        } else if (ps[k].find("EnsBufs") != std::string::npos) {
            const void* b[6];
            std::memcpy(b, args[k], sizeof b);
            for (const void* p : b)
                if (p && !room(p)) fail(sig + ": a table of EnsBufs is not live");
        }
    }
    if (items) {
        if (cfg_g.x == 0) fail(sig + ": empty grid");
        const int n = qoff[8];
        if (n <= 0 || room(items) < (size_t)n * sizeof(Item)) fail(sig + ": items");
        int pairs = 0;
        for (int t = 0; t < n; ++t) {
            const Item& w = items[t];
            if (w.off < 0 || w.off + 1 + w.nst > particles || w.j1 > w.off + 1 + w.nst ||
                (size_t)(w.pslot + w.nst) * 128 > part)
                fail(sig + ": an item of another state");
            pairs += w.ib == 0 ? w.j1 - w.j0 : 0;
        }
        // every cluster's stars once (those of the states below)
        if (particles && pairs <= 0) fail(sig + ": no items");
    }
}

}  // namespace

extern "C" {
void** __hipRegisterFatBinary(const void*)
{
    static void* h;
    return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* stub, char*, const char* name, unsigned, uint3*,
                           uint3*, dim3*, dim3*, int*)
{
    int st = 0;
    char* d = abi::__cxa_demangle(name, nullptr, nullptr, &st);
    names()[stub] = d ? d : name;
    std::free(d);
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t s)
{
    cfg_g = g;
    cfg_b = b;
    cfg_sh = sh;
    cfg_s = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, hipStream_t* s)
{
    *g = cfg_g;
    *b = cfg_b;
    *sh = cfg_sh;
    *s = cfg_s;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t)
{
    launched.push_back(names()[f]);
    check(names()[f], args);
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) { return give(p, n); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return give(p, n); }
hipError_t hipFree(void* p) { return take(p); }
hipError_t hipHostFree(void* p) { return take(p); }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    if (room(d) < n) fail("copy past a live block");
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t)
{
    if (room(d) < n) fail("memset past a live block");
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int)
{
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t)
{
    *n = 8;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipGetSymbolAddress(void**, const void*) { return hipErrorNotSupported; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    *s = (hipStream_t)1;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t)
{
    return hipErrorNotSupported;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e)
{
    *e = (hipEvent_t)1;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.0f;
    return hipSuccess;
}
}

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

bool ran(const char* kernel)
{
    for (const std::string& s : launched)
        if (s.find(kernel) != std::string::npos) return true;
    return false;
}

void want(int rc, int expect, const std::string& what)
{
    if (rc != expect)
        fail(what + ": status " + std::to_string(rc) + ", expected " + std::to_string(expect));
}

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
