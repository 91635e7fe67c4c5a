// pn1_io.hpp -- states between the caller's AoS arrays and the SoA device
// buffers of libpn1, through a context's pinned stage.
//
// The host copies the caller's arrays into the stage as they are (and the
// results out of it), and one kernel reads or writes the stage over the bus
// and transposes: one launch in place of a copy per component, and the
// transposition off the host.  Nothing waits for the kernel that reads the
// stage: whoever writes it next on the host waits for the stream first.
// Large states are bound by the bus (53 GB/s each way) and the host's copies.
// Measured on MI355X, upload and download with a copy per component and two
// waits / with these: n = 257, 72 / 23 us; n = 4097, 148 / 39 us; n = 131073,
// 1650 / 1400 us.
#pragma once
#include "pn1_common.hpp"

namespace pn1dev {

// Thread t of each kernel takes doubles 2 t and 2 t + 1 of the stage: 16 bytes
// per lane on the bus.
//
// Stage {x [n][3], v [n][3], m [n]} -> dst (6 x cap) and m, unless null; x is
// taken as zero if `xzero`.  Clears zero[0, nz).
inline __global__ __launch_bounds__(WG) void k_put(const double2* __restrict__ stage, int n,
                                                  size_t cap, bool xzero,
                                                  double* __restrict__ dst,
                                                  double* __restrict__ m,
                                                  double* __restrict__ zero, size_t nz)
{
    const size_t t = (size_t)blockIdx.x * WG + threadIdx.x, n3 = 3 * (size_t)n;
    const size_t len = 2 * n3 + (m ? (size_t)n : 0);
    if (2 * t < len && !(xzero && 2 * t + 1 < n3)) {
        const double2 w = stage[t];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const size_t q = 2 * t + b, h = q >= n3 ? 1 : 0, u = q - h * n3, i = u / 3;
            if (q < 2 * n3 && !(xzero && !h))
                dst[(3 * h + (u - 3 * i)) * cap + i] = b ? w.y : w.x;
            else if (q >= 2 * n3 && q < len)
                m[q - 2 * n3] = b ? w.y : w.x;
        }
    }
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const size_t q = 2 * t + b;
        if (xzero && q < n3) dst[(q - 3 * (q / 3)) * cap + q / 3] = 0.0;
        if (q < nz) zero[q] = 0.0;
    }
}

// src (3 nv x cap, from its first star) -> stage, nv arrays [n][3], then
// extra[0, ne).  The stage holds a whole number of double2.
inline __global__ __launch_bounds__(WG) void k_get(const double* __restrict__ src, int n,
                                                  size_t cap, int nv,
                                                  const double* __restrict__ extra, size_t ne,
                                                  double2* __restrict__ stage)
{
    const size_t t = (size_t)blockIdx.x * WG + threadIdx.x, n3 = 3 * (size_t)n;
    const size_t len = nv * n3 + ne;
    if (2 * t >= len) return;
    double w[2] = {0.0, 0.0};
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const size_t q = 2 * t + b, h = q >= n3 ? 1 : 0, u = q - h * n3, i = u / 3;
        if (q < nv * n3)
            w[b] = src[(3 * h + (u - 3 * i)) * cap + i];
        else if (q < len)
            w[b] = extra[q - nv * n3];
    }
    stage[t] = make_double2(w[0], w[1]);
}

// dst = src, both 6 x cap, stars 0 .. n - 1 (grid: 6 rows).
inline __global__ __launch_bounds__(WG) void k_copy6(const double* __restrict__ src, int n,
                                                    size_t cap, double* __restrict__ dst)
{
    const size_t i = (size_t)blockIdx.x * WG + threadIdx.x;
    if (i < (size_t)n) dst[blockIdx.y * cap + i] = src[blockIdx.y * cap + i];
}

}  // namespace pn1dev
