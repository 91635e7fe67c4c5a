// pn1_rows.hpp -- what the O(n) kernels of libpn1 (force and adjoint) share:
// rows of stars, their sums over a wave, and the sums over all rows by the
// last workgroup of a launch.
#pragma once
#include "pn1_common.hpp"

namespace pn1dev {

// ---------------------------------------------------------------------
// rows: the O(n) kernels take the stars in rows of 64 (one per lane of a
// wave), FG waves to a workgroup
// ---------------------------------------------------------------------
constexpr int RB = 64;
constexpr int FG = 8;
constexpr int FWG = FG * RB;
// A row's share of the sums over all stars: RV doubles, the BH's 1PN
// acceleration (3), then the NGS separable sums of the next evaluation.
constexpr int RV = 16;
constexpr int RV_G = 3;
static_assert(RV_G + NGS <= RV, "a row's values");

// Sum over the wave, in every lane (xor butterfly: the same bits in each).
__device__ __forceinline__ double wave_sum(double t)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
    return t;
}

// lo = {a in the lower half (G = 32) or the even rows of 16 (G = 16), b's
// other half moved there}, and hi the rest: adding both sums a over lane
// pairs l, l ^ G in the lanes without that bit and b in the others.
template <int G>
__device__ __forceinline__ double swap_sum(double a, double b)
{
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    const unsigned long long ua = (unsigned long long)__double_as_longlong(a);
    const unsigned long long ub = (unsigned long long)__double_as_longlong(b);
    u32x2 l, h;
    if (G == 32) {
        l = __builtin_amdgcn_permlane32_swap((unsigned)ua, (unsigned)ub, false, false);
        h = __builtin_amdgcn_permlane32_swap((unsigned)(ua >> 32), (unsigned)(ub >> 32), false, false);
    } else {
        l = __builtin_amdgcn_permlane16_swap((unsigned)ua, (unsigned)ub, false, false);
        h = __builtin_amdgcn_permlane16_swap((unsigned)(ua >> 32), (unsigned)(ub >> 32), false, false);
    }
    const double x = __longlong_as_double((long long)(((unsigned long long)h[0] << 32) | l[0]));
    const double y = __longlong_as_double((long long)(((unsigned long long)h[1] << 32) | l[1]));
    return x + y;
}

// A value that is the same in all lanes, in scalar registers.
__device__ __forceinline__ double to_scalar(double v)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)u);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// v of lane l ^ X, X = 1, 2, 4 or 8, by DPP (a ds_bpermute shuffle takes over 100 cycles).
template <int X>
__device__ __forceinline__ int lane_xor(int v)
{
    if (X == 1) return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true);      // quad 1 0 3 2
    if (X == 2) return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true);      // quad 2 3 0 1
    if (X == 8) return __builtin_amdgcn_mov_dpp(v, 0x128, 0xF, 0xF, true);     // row_ror 8
    v = __builtin_amdgcn_mov_dpp(v, 0x141, 0xF, 0xF, true);                    // l ^ 7, then
    return __builtin_amdgcn_mov_dpp(v, 0x1B, 0xF, 0xF, true);                  // quad 3 2 1 0
}
template <int X>
__device__ __forceinline__ double lane_xor(double v)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)lane_xor<X>((int)(unsigned)u);
    const unsigned hi = (unsigned)lane_xor<X>((int)(unsigned)(u >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// The wave's sums of 16 values: lane l gets the sum of v[l >> 2] over all
// lanes.  Halving the values at each exchange takes 15 of them instead of
// the 16 x 6 of one butterfly per value, and half the code, which in kernels
// that run each instruction once is most of their time.
__device__ __forceinline__ double wave_sums16(const double (&v)[16])
{
    const int lane = threadIdx.x & 63;
    double a[8], b[4], c[2];
#pragma unroll
    for (int k = 0; k < 8; ++k) a[k] = swap_sum<32>(v[k], v[8 + k]);
#pragma unroll
    for (int k = 0; k < 4; ++k) b[k] = swap_sum<16>(a[k], a[4 + k]);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const bool up = lane & 8;
        const double keep = up ? b[2 + k] : b[k], send = up ? b[k] : b[2 + k];
        c[k] = keep + lane_xor<8>(send);
    }
    const bool up = lane & 4;
    double t = (up ? c[1] : c[0]) + lane_xor<4>(up ? c[0] : c[1]);
    t += lane_xor<2>(t);
    t += lane_xor<1>(t);
    return t;
}

// The same over the lower 16 lanes: lane l < 16 gets the sum of v[l].
template <int X, int N>
__device__ __forceinline__ void halve(const double (&v)[2 * N], double (&o)[N])
{
    const bool up = threadIdx.x & X;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const double keep = up ? v[N + k] : v[k], send = up ? v[k] : v[N + k];
        o[k] = keep + lane_xor<X>(send);
    }
}
__device__ __forceinline__ double group_sums16(const double (&v)[16])
{
    double a[8], b[4], c[2], d[1];
    halve<8>(v, a);
    halve<4>(a, b);
    halve<2>(b, c);
    halve<1>(c, d);
    return d[0];
}

// Values that one workgroup hands to another within a launch (the rows' sums
// and masks, to the last workgroup): stored and loaded at device scope, past
// the XCD's own L2.  A release fence would do the same for ordinary stores,
// but it writes back every dirty line of that L2, per workgroup (measured on
// MI355X: 0.14 us each, 1.4 ms of an ensemble's 9864 workgroups).
template <typename T>
__device__ __forceinline__ void hand_over(T* p, T v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ T take_over(const T* p)
{
    return __hip_atomic_load(const_cast<T*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Fixed-order sums of rows [b0, b1), by a workgroup of FWG threads, into
// tot[RV] (LDS), for every thread of it: thread t adds value t % RV of rows
// t / RV, t / RV + FWG / RV, ...  Q: the values are those of a row's Q groups
// of 16 stars.
template <int Q = 1>
__device__ __forceinline__ void rows_total(const double* rows, int b0, int b1, double* tot)
{
    __shared__ double sh[FG][RV];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    double t = 0.0;
    if (Q == 1) {
#pragma unroll 8
        for (int b = b0 + (int)threadIdx.x / RV; b < b1; b += FWG / RV)
            t += take_over(&rows[(size_t)b * RV + (threadIdx.x & (RV - 1))]);
    } else {
#pragma unroll 2
        for (int b = b0 + (int)threadIdx.x / RV; b < b1; b += FWG / RV) {
            const double* r = &rows[(size_t)b * 4 * RV + (threadIdx.x & (RV - 1))];
            t += (take_over(r) + take_over(r + RV)) + (take_over(r + 2 * RV) + take_over(r + 3 * RV));
        }
    }
    t += __shfl_xor(t, 16, 64);
    t += __shfl_xor(t, 32, 64);
    if (lane < RV) sh[wid][lane] = t;
    __syncthreads();
    if (threadIdx.x < RV) {
        t = sh[0][threadIdx.x];
#pragma unroll
        for (int w = 1; w < FG; ++w) t += sh[w][threadIdx.x];
        tot[threadIdx.x] = t;
    }
    __syncthreads();
}

// Whether this workgroup is the last of `nblk` to get here (the counter goes
// back to 0 for the next launch).  What the others handed over before is
// visible to it: every wave waits for its own stores to complete before the
// workgroup takes its ticket, and the last ticket is taken after all others.
// Every thread of the workgroup calls it.
__device__ __forceinline__ bool last_block(unsigned int* cnt, unsigned int nblk)
{
    __shared__ bool s_last;
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned int t =
            __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = t == nblk - 1;
        if (s_last) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    return s_last;
}

}  // namespace pn1dev
