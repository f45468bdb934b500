// B-spline weights and grid coordinates shared by the spreading, gathering and
// solver kernels (computeBSplinePoint and computeMPIDBsplines,
// MPIDReferenceForce.cpp:2956-3075).
#pragma once

#include "engine.h"

namespace mpid {

// Order-6 B-spline weights of the 6 grid points and their first ND derivatives:
// Cox-de Boor recursion, derivatives as backward differences of lower orders.
template <class R, int ND>
__device__ __forceinline__ void bspline6(R w, R th[kOrder][ND + 1]) {
    R c[kOrder + 1][kOrder + 1];
    c[1][0] = R(1);
#pragma unroll
    for (int p = 2; p <= kOrder; p++) {
#pragma unroll
        for (int m = 0; m < p; m++) {
            R left = (m >= 1) ? c[p - 1][m - 1] : R(0);
            R right = (m <= p - 2) ? c[p - 1][m] : R(0);
            c[p][m] = ((w + R(p - 1 - m)) * left + (R(m + 1) - w) * right) * R(1.0 / (p - 1));
        }
    }
#pragma unroll
    for (int r = 0; r <= ND; r++) {
        R cur[kOrder + 1];
        const int p = kOrder - r;
#pragma unroll
        for (int m = 0; m < kOrder + 1; m++) cur[m] = (m < p) ? c[p][m] : R(0);
        int len = p;
#pragma unroll
        for (int s = 0; s < r; s++) {
            R nxt[kOrder + 1];
#pragma unroll
            for (int m = 0; m < kOrder + 1; m++)
                nxt[m] = ((m >= 1 && m - 1 < len) ? cur[m - 1] : R(0)) - ((m < len) ? cur[m] : R(0));
            len++;
#pragma unroll
            for (int m = 0; m < kOrder + 1; m++) cur[m] = nxt[m];
        }
#pragma unroll
        for (int m = 0; m < kOrder; m++) th[m][r] = cur[m];
    }
}

__device__ __forceinline__ unsigned spread_bits_pme(unsigned v) {
    v &= 0x3ffu;
    v = (v | (v << 16)) & 0x030000ffu;
    v = (v | (v << 8)) & 0x0300f00fu;
    v = (v | (v << 4)) & 0x030c30c3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

// Grid origin and spline offset of one atom along an axis of n points from
// its fractional coordinate f along that box vector, as the reference
// computes them (f wrapped to [-1/2, 1/2), then shifted by one half box,
// MPIDReferenceForce.cpp:3049-3075).
template <class R>
__device__ __forceinline__ void grid_coord(R f, int n, int& ig, R& w) {
    f -= floor(f + R(0.5));
    const R fr = R(n) * (f + R(0.5));
    const int ifr = (int)floor(fr);
    w = fr - R(ifr);
    ig = ifr - kOrder + 1;
    ig %= n;
    if (ig < 0) ig += n;
}

// Row k of a spline table, by unrolled compares (a dynamically indexed
// register array would go to scratch memory).
template <class R, int ND>
__device__ __forceinline__ void spline_at(const R (&t)[kOrder][ND + 1], int k, R (&out)[ND + 1]) {
#pragma unroll
    for (int d = 0; d <= ND; d++) out[d] = t[0][d];
#pragma unroll
    for (int m = 1; m < kOrder; m++)
        if (k == m) {
#pragma unroll
            for (int d = 0; d <= ND; d++) out[d] = t[m][d];
        }
}

}  // namespace mpid
