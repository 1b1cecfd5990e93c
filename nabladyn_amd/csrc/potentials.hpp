// Pair potentials as device functors: each maps a pair's squared distance (below the cutoff)
// to its energy u and to fs = -(du/dr)/r, so that the force on i from j is fs * r_ij.
//
// LJ: u = 4 eps [(s2/r2)^6 - (s2/r2)^3] - u_c with u_c the same at rc
//     (potential/_lennard_jones/_potential.py:113-120,209-234).
// Table: Catmull-Rom on knots padded with a virtual knot at each end and the last knot read as 0;
//     below the first knot the row's tangent there (potential/_tabulated/_potential.py:59-91).
#pragma once

#include "common.hpp"

namespace ndn {

// 1 / value: the hardware reciprocal in fp32 (1 ulp); in fp64 the hardware's estimate with two
// Newton steps, whose result is the correctly rounded one but next to a rounding boundary, in half
// the instructions of a division (which also scales operands near the ends of the range). For
// factors that only scale a force. Zero gives NaN in fp64, where its caller's terms are NaN too.
template <typename T>
__device__ __forceinline__ T reciprocal(T value);
template <>
__device__ __forceinline__ float reciprocal<float>(float value)
{
    return __builtin_amdgcn_rcpf(value);
}
template <>
__device__ __forceinline__ double reciprocal<double>(double value)
{
    double y = __builtin_amdgcn_rcp(value);
    y = __builtin_fma(__builtin_fma(-value, y, 1.0), y, y);
    return __builtin_fma(__builtin_fma(-value, y, 1.0), y, y);
}

// sqrt(x), correctly rounded: the hardware's reciprocal square root with a coupled Newton step (two
// in fp64) and a last one on the remainder (P. W. Markstein, "Computation of elementary
// functions on the IBM RISC System/6000 processor", 1990), without the scaling that a library's
// root does for results near the ends of the range: squared distances are far from them, and one
// that is not takes the hardware's root.
template <typename T>
__device__ __forceinline__ T pair_distance(T x);
template <>
__device__ __forceinline__ double pair_distance<double>(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    return x > 1e-200 ? g : __builtin_amdgcn_sqrt(x);
}
template <>
__device__ __forceinline__ float pair_distance<float>(float x)
{
    const float y = __builtin_amdgcn_rsqf(x);
    float g = x * y, h = 0.5f * y;
    const float r = __builtin_fmaf(-h, g, 0.5f);
    g = __builtin_fmaf(g, r, g);
    h = __builtin_fmaf(h, r, h);
    g = __builtin_fmaf(__builtin_fmaf(-g, g, x), h, g);
    return x > 1e-30f ? g : __builtin_amdgcn_sqrtf(x);
}

// 1 / x: the hardware reciprocal with one Newton step in fp32, two in fp64.
template <typename T>
__device__ __forceinline__ T refined_reciprocal(T x);
template <>
__device__ __forceinline__ double refined_reciprocal<double>(double x)
{
    return reciprocal(x);
}
template <>
__device__ __forceinline__ float refined_reciprocal<float>(float x)
{
    const float y = __builtin_amdgcn_rcpf(x);
    const float better = __builtin_fmaf(__builtin_fmaf(-x, y, 1.0f), y, y);
    // the step makes NaN of the ends of the range (0, infinity), whose reciprocals are exact
    return better == better ? better : y;
}

// Row of the unordered type pair (a, b): a(2T - a - 1)/2 + b for a <= b
// (potential/_lennard_jones/_potential.py:143-151).
__device__ __forceinline__ int pair_row(std::int64_t a, std::int64_t b, int num_types)
{
    const std::int64_t low = a < b ? a : b;
    const std::int64_t high = a < b ? b : a;
    return static_cast<int>(low * (2 * num_types - low - 1) / 2 + high);
}

// Per-row LJ coefficients, built once per evaluation by a prologue kernel.
template <typename T>
struct LJRow
{
    T sigma_squared;
    T four_eps;
    T twentyfour_eps;
    T shift;
};

template <typename T>
struct LJ
{
    const LJRow<T>* __restrict__ rows;
    const std::int64_t* __restrict__ types;
    int num_types;

    __device__ __forceinline__ int row(std::int64_t i, std::int64_t j) const
    {
        return num_types == 1 ? 0 : pair_row(types[i], types[j], num_types);
    }

    __device__ __forceinline__ void eval(int row_index, T r2, T& u, T& fs) const
    {
        const LJRow<T> c = rows[row_index];
        // 1/r^2 by the hardware reciprocal (1 ulp in fp32), as the MD kernels take it
        const T inverse = reciprocal(r2);
        const T s = c.sigma_squared * inverse;
        const T p6 = s * s * s;
        u = c.four_eps * (p6 * p6 - p6) - c.shift;
        fs = c.twentyfour_eps * (T(2) * p6 * p6 - p6) * inverse;
    }
};

// The padded table of a row: [K + 2] knots, the last real knot 0, virtual knots at both ends.
template <typename T>
struct Table
{
    const T* __restrict__ padded;        // [P, K + 2]
    const T* __restrict__ start;         // [P]
    const T* __restrict__ spacing;       // [2, P]: the spacings, then 1 / spacing
    const std::int64_t* __restrict__ types;
    int num_types;
    int knots;                           // K

    __device__ __forceinline__ int row(std::int64_t i, std::int64_t j) const
    {
        return num_types == 1 ? 0 : pair_row(types[i], types[j], num_types);
    }

    __device__ __forceinline__ void eval(int row_index, T r2, T& u, T& fs) const
    {
        // r and the knot coordinate are the reference's: its square root, subtraction and
        // division, each correctly rounded (pair_distance; the quotient is a product with 1/h
        // corrected by its remainder, which is the quotient's rounding when 1/h is correctly
        // rounded itself, as a hardware reciprocal with Newton steps is not for every h), so t
        // and the segment are the reference's bits
        const T r = pair_distance(r2);
        const T h = spacing[row_index];
        const T inverse_h = spacing[num_types * (num_types + 1) / 2 + row_index];
        const T offset = r - start[row_index];
        const T q = offset * inverse_h;
        const T x = fma(fma(-q, h, offset), inverse_h, q);
        T segment = floor(x);
        segment = segment < T(0) ? T(0) : (segment > T(knots - 2) ? T(knots - 2) : segment);
        const T t = x - segment;
        const T* k = padded + static_cast<std::int64_t>(row_index) * (knots + 2) +
                     static_cast<int>(segment);
        const T u0 = k[0], u1 = k[1], u2 = k[2], u3 = k[3];
        const T a = u2 - u0;
        const T b = T(2) * u0 - T(5) * u1 + T(4) * u2 - u3;
        const T c = T(3) * (u1 - u2) + u3 - u0;
        const T s = t > T(0) ? t : T(0);
        const T cubic = u1 + T(0.5) * s * (a + s * (b + s * c));
        const bool below = t < T(0);
        u = cubic + (below ? T(0.5) * a * t : T(0));
        const T du_dt = below ? T(0.5) * a : T(0.5) * (a + s * (T(2) * b + T(3) * s * c));
        // 1/r only scales the force: the hardware's reciprocal
        fs = -(du_dt * inverse_h) * reciprocal(r);
    }
};

}  // namespace ndn
