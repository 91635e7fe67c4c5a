// A HIP runtime over host memory, for CPU checks of libpn1's host code: the
// entry points that libpn1.so calls.  Allocations are registered (and only
// marked dead when freed), one of them can be refused, and a launch, which runs
// nothing, has its arguments checked instead: every pointer (also those of
// EnsBufs) must lie in a live allocation, and the work items a pair kernel gets
// must be the state's.  An executable that includes this and exports its
// symbols takes the library's calls.
#pragma once
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>


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
float (*elapsed)() = [] { return 1.0f; };      // of the launches since the last call
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
    *ms = elapsed();
    return hipSuccess;
}
}

namespace {

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
