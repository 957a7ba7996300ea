// fb_points.h -- device helpers over a field's points and values, shared between translation units.
#pragma once

#include "fb_internal.h"

namespace fb {

// min, max and a NaN flag of v[k] for k = k0, k0 + step, ... < k1, the loads of eight steps
// issued before their first use (one thread's share of a workgroup's values)
__device__ __forceinline__ void minmax_range(const double *__restrict__ v, int64_t k0, int64_t k1, int step,
                                             double &mn, double &mx, int &isn)
{
    constexpr int kUnroll = 8;
    int64_t k = k0;
    for (; k + (kUnroll - 1) * step < k1; k += kUnroll * step) {
        double x[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) x[u] = v[k + u * step];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            if (x[u] != x[u]) isn = 1;
            mn = fmin(mn, x[u]);
            mx = fmax(mx, x[u]);
        }
    }
    for (; k < k1; k += step) {
        const double x = v[k];
        if (x != x) isn = 1;
        mn = fmin(mn, x);
        mx = fmax(mx, x);
    }
}

// (min, max, NaN flag) of the wave's lanes, in every lane
__device__ __forceinline__ void minmax_wave(double &mn, double &mx, int &isn)
{
    for (int d = 32; d >= 1; d >>= 1) {
        mn = fmin(mn, __shfl_xor(mn, d));
        mx = fmax(mx, __shfl_xor(mx, d));
    }
    isn = __any(isn);
}

__device__ __forceinline__ double field_offset(double mn, double mx, int isn)
{
    return isn ? __builtin_nan("") : (mn + mx) / 2.0;
}

// Zero fill of z by workgroups of THREADS threads, PER 16-byte words each: workgroup b of the
// remaining ranges fills its share if it lies in z; else b moves on past z.
template <int THREADS, int PER>
__device__ __forceinline__ bool zero_block(const ZeroRange &z, int64_t &b)
{
    constexpr int64_t per = THREADS * PER;
    const int64_t nb = (z.n + per - 1) / per;
    if (b >= nb) {
        b -= nb;
        return false;
    }
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int64_t i = b * per + k * THREADS + threadIdx.x;
        if (i < z.n) z.p[i] = make_uint4(0u, 0u, 0u, 0u);
    }
    return true;
}

template <int THREADS, int PER>
inline int64_t zero_blocks(const ZeroRange &z)
{
    return (z.n + THREADS * PER - 1) / (THREADS * PER);
}

// grid position of a point: xc = (p - x0)/step per axis, dropped when outside
// [0, size-1) on any axis (interpolation.py:247-250).  NaN coordinates are
// dropped as well (the reference's int(NaN) is undefined).

struct PointPos {
    int64_t i[3];
    double w[3];
};

__device__ __forceinline__ bool point_pos(const FieldDev &F, const double *__restrict__ p, PointPos &pp)
{
    bool inside = true;
    for (int m = 0; m < 3; ++m) {
        pp.i[m] = 0;
        pp.w[m] = 0.0;
    }
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        if (m < F.dim) {
            const double c = (p[m] - F.x0[m]) / F.step[m];
            if (!(c >= 0.0) || c >= (double)(F.size[m] - 1)) inside = false;
            const int64_t ci = inside ? (int64_t)c : 0;
            pp.i[m] = ci;
            pp.w[m] = c - (double)ci;
        }
    }
    return inside;
}

}  // namespace fb
