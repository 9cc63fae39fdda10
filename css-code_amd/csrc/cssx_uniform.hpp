// The compact solve with constant coefficients (gfx950), used by the sweeps of pencils long
// enough that their two ends do not see each other.
//
// Away from the closure rows every row of the tridiagonal system is  al x_{j-1} + x_j + al x_{j+1} = d_j.
// With the pivot p = (1 + sqrt(1 - 4 al^2))/2 that elimination converges to, and a = al/p, that matrix
// factors into two first-order recurrences with constant coefficients,
//   y_j = d_j/p - a y_{j-1}        x_j = y_j - a x_{j+1},
// exactly, but for the first row, whose diagonal entry becomes p instead of 1.  Starting the
// recurrence with y = 0 above row b therefore solves a system that differs from the true one only in
// row b, and the difference is a multiple of (-a)^(j-b) (the decaying solution of the homogeneous
// rows): a correction known once x_b is (lower_end below).  An unknown above the last uniform
// row enters the same way from the other side, as the carry x_{j+1} of the backward recurrence
// (upper_end).  So neither end needs coefficients of its own along the pencil.
//
// A pencil cut into segments solves each with zero carry-in; a carry Y from below adds
// (-a)^(j+1) Y to row j and a carry X from above (-a)^(m-j) X.  a = 0.382 (first derivative) and 0.188
// (second): a carry is below an eighth of the rounding of the type (a^reach < 2^-27, 2^-55) `reach` rows on, so it
// spans the next one to few segments only and needs no reduced system.
//
// What that means for results: an error is small against the largest value within `reach` rows or so, not against
// a much smaller value there (the tail of a spike ends about `reach` rows from it instead of decaying on), and a NaN or
// an infinity fills that reach and the rest of the segments or lanes it meets (up to 55 rows either way in FP32, 81 in
// FP64), not the whole pencil.
#pragma once
#include <hip/hip_runtime.h>

#include "cssx_kernels.hpp"
#include "cssx_rows.hpp"

namespace cssx {

template <int ORDER>
struct Uni;
template <>
struct Uni<1> {
    static constexpr double al = 1.0 / 3.0, p = 0.87267799624996494940, a = 0.38196601125010515180;
    static constexpr double l1 = 0.125, u1 = 0.75;   // closure row 1: l1 x_0 + x_1 + u1 x_2
    static constexpr int reach32 = 20, reach64 = 40;
};
template <>
struct Uni<2> {
    static constexpr double al = 2.0 / 11.0, p = 0.96577048936179992651, a = 0.18826230851010040420;
    static constexpr double l1 = 0.1, u1 = -0.35;
    static constexpr int reach32 = 12, reach64 = 24;
};
// (-a)^k
template <int ORDER>
__host__ __device__ constexpr double uni_pow(int k) {
    double v = 1.0;
    for (int i = 0; i < (k < 0 ? -k : k); i++) v *= -Uni<ORDER>::a;
    return k < 0 ? 1.0 / v : v;
}
// rows after which a carry is below the rounding of T
template <typename T, int ORDER>
constexpr int uni_reach() {
    constexpr int r = sizeof(T) == 4 ? Uni<ORDER>::reach32 : Uni<ORDER>::reach64;
    static_assert(r % 2 == 0 && uni_pow<ORDER>(r) < (sizeof(T) == 4 ? 0x1p-27 : 0x1p-55), "a carry is cut too early");
    return r;
}
// The first wall row's coefficient of x_1 (cssx_plan.cpp lhs_coefficients) and the reciprocal of the
// eliminated wall system's pivot, by closure kind; compile-time constants, selected per launch.
template <int ORDER>
struct UniWall {
    static constexpr double u0d = ORDER == 1 ? 4.0 : 137.0 / 13.0, u0n = ORDER == 1 ? 0.0 : 707.0 / 193.0;
    static constexpr double invd = 1.0 / (1.0 - Uni<ORDER>::l1 * u0d - Uni<ORDER>::u1 * Uni<ORDER>::a);
    static constexpr double invn = 1.0 / (1.0 - Uni<ORDER>::l1 * u0n - Uni<ORDER>::u1 * Uni<ORDER>::a);
};

// right-hand sides of the two wall rows at the lower (HI = false) or upper end, f[k] the k-th point from
// the wall, val the prescribed wall derivative in index units; times `scale`
template <typename T, int ORDER, bool HI>
__device__ __forceinline__ void wall_rhs(const T (&f)[6], int bd, T val, T scale, T &r0, T &r1) {
    const bool dirichlet = HI ? (bd == 1 || bd == 2) : (bd == 1 || bd == 3);
    if constexpr (ORDER == 1) {
        const T s1 = Rows<T, 1>::wall1(f[0], f[1], f[2], f[3], f[4]);
        const T s0 = Rows<T, 1>::wall0(dirichlet, (HI ? (bd == 3 || bd == 4) : bd != 0) ? val : T(0), f[0], f[1], f[2],
                                       f[3], s1);
        r1 = HI ? -s1 : s1;
        r0 = (HI && dirichlet) ? -s0 : s0;
    } else {
        const T v = bd == 0 ? T(0) : (HI ? val : -val);
        r1 = Rows<T, 2>::wall1(f[0], f[1], f[2], f[3], f[4]);
        r0 = Rows<T, 2>::wall0(dirichlet, v, f[0], f[1], f[2], f[3], f[4], f[5]);
    }
    r0 *= scale;
    r1 *= scale;
}

// Lower wall: from x'_2 (the uniform solve's row 2) the solution's rows 0, 1 and the factor s of
// the correction s (-a)^(j-2) of rows j >= 2:
//   x_0 + u0 x_1 = r0,  l1 x_0 + x_1 + u1 x_2 = r1,  x_2 = x'_2 + s,  al x_1 + (1-p) x'_2 + p s = 0
template <typename T, int ORDER>
__device__ __forceinline__ T lower_wall(T x2, T r0, T r1, bool dirichlet, T &x0, T &x1) {
    using U = Uni<ORDER>;
    using V = UniWall<ORDER>;
    const T u0 = dirichlet ? (T)V::u0d : (T)V::u0n, inv = dirichlet ? (T)V::invd : (T)V::invn;
    x1 = (r1 - (T)U::l1 * r0 - (T)(U::u1 * (1.0 - U::a * U::a)) * x2) * inv;
    x0 = r0 - u0 * x1;
    return (T)(-U::a) * x1 - (T)(U::a * U::a) * x2;
}
// Upper wall: from y of row n-3 the solution's rows n-2 and n-1
template <typename T, int ORDER>
__device__ __forceinline__ void upper_wall(T y3, T r0, T r1, bool dirichlet, T &xn2, T &xn1) {
    using U = Uni<ORDER>;
    using V = UniWall<ORDER>;
    const T u0 = dirichlet ? (T)V::u0d : (T)V::u0n, inv = dirichlet ? (T)V::invd : (T)V::invn;
    xn2 = (r1 - (T)U::l1 * r0 - (T)U::u1 * y3) * inv;
    xn1 = r0 - u0 * xn2;
}

// Interior right-hand side of the forward recurrence, d_j/p times `scale`, from rows j-2 .. j+2.  Each
// constant is rounded once (a product of rounded factors would bias every row of the sweep the
// same way: 6.9e-8 against 1.4e-7 relative error in FP32).
template <typename T, int ORDER>
struct Stencil {
    T c1, c2, c0;
    __device__ __forceinline__ explicit Stencil(T scale) {
        constexpr double p = Uni<ORDER>::p;
        c1 = (T)((double)scale * ((ORDER == 1 ? 7.0 / 9.0 : 12.0 / 11.0) / p));
        c2 = (T)((double)scale * ((ORDER == 1 ? 1.0 / 36.0 : 3.0 / 44.0) / p));
        c0 = (T)((double)scale * (1.0 / p));   // of a row assembled elsewhere
    }
    __device__ __forceinline__ T operator()(T m2, T m1, T x0, T p1, T p2) const {
        if constexpr (ORDER == 1) return c1 * (p1 - m1) + c2 * (p2 - m2);
        else return c1 * (p1 - T(2) * x0 + m1) + c2 * (m2 - T(2) * x0 + p2);
    }
};

}  // namespace cssx
