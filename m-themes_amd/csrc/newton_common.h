// newton_common.h -- what the loop's stress update (newton.hip) and the batch's
// (newton_batch.hip) share: integral powers and the change of basis.
#pragma once

#include "evpgpu_impl.h"

namespace {

__device__ __forceinline__ double ipow(double x, int m)
{
    double r = 1.0, b = x;
    while (m) {
        if (m & 1) r *= b;
        b *= b;
        m >>= 1;
    }
    return r;
}

// x^m for a wave-uniform 0 <= m < 32: the products of ipow in the same
// order, straight-line (a scalar-masked select per exponent bit instead of a
// scalar loop, whose instructions and branches cost issue slots)
__device__ __forceinline__ double ipow5(double x, int m)
{
    double r = 1.0, b = x;
#pragma unroll
    for (int i = 0; i < 5; i++) {
        const double t = r * b;
        r = ((m >> i) & 1) ? t : r;
        if (i < 4) b *= b;
    }
    return r;
}

// chg_basis opt 2 for a symmetric tensor given as (11 22 33 23 13 12)
__device__ __forceinline__ void sym_to_v6(const double t[6], double v[6])
{
    const double r2 = RSQ2, r3 = RSQ3, r6 = RSQ6;
    v[0] = t[0] * (-1. * r2) + t[1] * r2;
    v[1] = t[0] * (-1. * r6) + t[1] * (-1. * r6) + t[2] * (2. * r6);
    v[2] = t[3] * r2 + t[3] * r2;
    v[3] = t[4] * r2 + t[4] * r2;
    v[4] = t[5] * r2 + t[5] * r2;
    v[5] = t[0] * r3 + t[1] * r3 + t[2] * r3;
}

// chg_basis opt 1 -> symmetric (11 22 33 23 13 12)
__device__ __forceinline__ void v6_to_sym(const double v[6], double t[6])
{
    const double r2 = RSQ2, r3 = RSQ3, r6 = RSQ6;
    t[0] = v[0] * (-1. * r2) + v[1] * (-1. * r6) + v[5] * r3;
    t[1] = v[0] * r2 + v[1] * (-1. * r6) + v[5] * r3;
    t[2] = v[1] * (2. * r6) + v[5] * r3;
    t[3] = v[2] * r2;
    t[4] = v[3] * r2;
    t[5] = v[4] * r2;
}

} // namespace
