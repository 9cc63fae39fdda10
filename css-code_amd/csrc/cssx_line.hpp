// One pencil along the lanes of a wavefront: loads, the constant-coefficient compact solve
// (cssx_uniform.hpp) and stores of a unit-stride pencil whose lane j holds rows [j*MR, j*MR + MR).
// Several pencils sit side by side in a wavefront; lanes past the last pencil take part with zeros.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "cssx_bufio.hpp"
#include "cssx_uniform.hpp"

namespace cssx {

// REM = n mod MR, which makes the last lane's row count m and the place kn2 of row n-2 compile-time; -1: known
// at run time only (n and nl are wave-uniform, so the comparisons with a row number k below are scalar).
template <int MR, int REM>
struct LineShape {
    static constexpr bool FULL = REM == 0;   // every lane holds MR rows
    int n, nl, j, m;      // pencil rows, lanes per pencil, this lane, rows of the last lane
    int jn2, kn2;         // lane and position of row n-2
    bool active, first, last, at_n2;
    __device__ __forceinline__ LineShape(int n_, int nl_, int j_, bool act) : n(n_), nl(nl_), j(j_), active(act) {
        if constexpr (REM >= 0) {
            m = REM == 0 ? MR : REM;
            kn2 = (REM + MR - 2) % MR;
            jn2 = REM == 1 ? nl - 2 : nl - 1;
        } else {
            m = n - (nl - 1) * MR;
            kn2 = (n - 2) % MR;
            jn2 = (n - 2) / MR;
        }
        first = act && j == 0;
        last = act && j == nl - 1;
        at_n2 = act && j == jn2;
    }
    template <typename T>
    __device__ __forceinline__ T pick(const T (&v)[MR], int k0) const {
        T r = v[MR - 1];
#pragma unroll
        for (int k = 0; k < MR - 1; k++) {
            const T t = v[k];   // (read first: a conditional read would index the array in scratch)
            r = k == k0 ? t : r;
        }
        return r;
    }
};

// MR values at p + at as 16-byte loads (4-byte alignment); a lane whose run leaves the `total` values
// there (the last lane of the last pencil) reads them one by one.  Rows past the pencil's end belong to the
// next pencil: the caller's rows beyond n-1 are not used.
template <typename T, int MR, int REM>
__device__ __forceinline__ void line_load(const T *__restrict__ p, long at, long total, const LineShape<MR, REM> &G,
                                          T (&v)[MR]) {
#pragma unroll
    for (int k = 0; k < MR; k++) v[k] = T(0);
    if (!G.active) return;
    if (REM == 0 || at + MR <= total) {
        __builtin_memcpy(v, p + at, sizeof(v));
    } else {
#pragma unroll
        for (int k = 0; k < MR; k++)
            if (at + k < total) v[k] = p[at + k];
    }
}

// (`at` long, or unsigned from a base that is the same for the wavefront: a 32-bit lane offset in bytes)
template <typename T, int MR, int REM, class I>
__device__ __forceinline__ void line_store(T *__restrict__ p, I at, const LineShape<MR, REM> &G, const T (&x)[MR]) {
    if (REM == 0 || !G.last || G.m == MR) {
        __builtin_memcpy((char *)p + at * (I)sizeof(T), x, sizeof(x));
        return;
    }
    // the last lane's m < MR rows in pieces of 8, 4, 2 and 1 (m is wave-uniform; one store per set bit)
    auto piece = [&](auto cnt, int from) {
        constexpr int C = decltype(cnt)::value;
#pragma unroll
        for (int f = 0; f + C <= MR; f += C)
            if (f == from) __builtin_memcpy((char *)p + (at + (I)f) * (I)sizeof(T), &x[f], C * sizeof(T));
    };
    int from = 0;
    if constexpr (MR > 8) {
        if (G.m & 8) piece(std::integral_constant<int, 8>{}, from), from += 8;
    }
    if (G.m & 4) piece(std::integral_constant<int, 4>{}, from), from += 4;
    if (G.m & 2) piece(std::integral_constant<int, 2>{}, from), from += 2;
    if (G.m & 1) piece(std::integral_constant<int, 1>{}, from);
}

// Pencils that stay within a wavefront pass nothing to its neighbours
struct LineWithin {
    static constexpr bool ON = false;
};
// Pencils cut by the end of a wavefront (lanes of a workgroup in one strip): what one side of the cut needs
// from the other goes through LDS, the six rows next to it for all fields at once and the carry of each
// recurrence per field, in words that one field and direction owns (one barrier per exchange, none to protect a
// word's reuse).  A carry dies before the far end of a wavefront, so the sender needs none of its own.
// The lanes are laid so that the cut is never within the first lanes of a pencil (its lower-wall
// correction stays in its wavefront) nor before its last lane (rows n-2 and n-1).
template <typename T, int NF, int NW>
struct LineCut {
    T rows[NF][NW][6], up[NF][NW], dn[NF][NW];
};
template <typename T, int MR, int NF, int NW>
struct LineAcross {
    static constexpr bool ON = true;
    LineCut<T, NF, NW> &L;
    int f, w, lane;          // field, wavefront, lane
    bool from_below, from_above;   // the lane belongs to a pencil cut at its wavefront's lower / upper end
    T q_below, q_above;      // (-a)^(rows between the cut and the lane)
    static __device__ __forceinline__ void barrier() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    }
    // posts the lane's edge rows of field k (a barrier follows)
    __device__ __forceinline__ void post(int k, const T (&v)[MR]) {
        if (lane == 63) {
#pragma unroll
            for (int i = 0; i < 4; i++) L.rows[k][w][i] = v[MR - 4 + i];
        }
        if (lane == 0) {
            L.rows[k][w][4] = v[0];
            L.rows[k][w][5] = v[1];
        }
    }
    __device__ __forceinline__ void window(T (&lo)[4], T (&hi)[2]) const {
        const int b = w > 0 ? w - 1 : 0, a = w < NW - 1 ? w + 1 : w;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const T t = L.rows[f][b][i];
            lo[i] = lane == 0 ? t : lo[i];
        }
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const T t = L.rows[f][a][4 + i];
            hi[i] = lane == 63 ? t : hi[i];
        }
    }
    __device__ __forceinline__ T carry_up(T out) {
        if (lane == 63) L.up[f][w] = out;
        barrier();
        const T t = L.up[f][w > 0 ? w - 1 : 0];
        return from_below ? q_below * t : T(0);
    }
    __device__ __forceinline__ T carry_down(T out) {
        if (lane == 0) L.dn[f][w] = out;
        barrier();
        const T t = L.dn[f][w < NW - 1 ? w + 1 : w];
        return from_above ? q_above * t : T(0);
    }
};

// The derivative of the wavefront's pencils (walls at both ends), times `scale`, in x; row n-1 comes back
// as the return value of the lane that holds row n-2 (see line_last).  lo_val / hi_val: the prescribed
// wall derivatives in index units, read on the lanes of rows 0 and n-2.  v's rows past n-1 are
// overwritten.
template <typename T, int ORDER, int MR, int REM, class X = LineWithin>
__device__ __forceinline__ T line_solve(const LineShape<MR, REM> &G, T (&v)[MR], int bd, T lo_val, T hi_val, T scale,
                                        T (&x)[MR], X cut = X()) {
    using U = Uni<ORDER>;
    // carries that reach `reach` rows span this many lanes
    constexpr int NT = (uni_reach<T, ORDER>() + MR - 1) / MR;
    constexpr T A = (T)U::a, Q = (T)uni_pow<ORDER>(MR);
    const int kn2 = G.kn2;
    // window: rows -4 .. MR+1 of the lane (two rows on either side for the stencil, two more below
    // for the upper closure)
    T lo[4], hi[2];
#pragma unroll
    for (int k = 0; k < 4; k++) lo[k] = from_prev(v[MR - 4 + k]);
    hi[0] = from_next(v[0]);
    hi[1] = from_next(v[1]);
    if constexpr (X::ON) cut.window(lo, hi);
    auto f = [&](int k) -> T { return k < 0 ? lo[k + 4] : k < MR ? v[k] : hi[k - MR]; };
    // ---- wall rows
    T r0 = T(0), r1 = T(0), q0 = T(0), q1 = T(0);
    {
        const T e[6] = {f(0), f(1), f(2), f(3), f(4), f(5)};
        wall_rhs<T, ORDER, false>(e, bd, lo_val, scale, r0, r1);
    }
#pragma unroll
    for (int k = 0; k < MR; k++)
        if (k == kn2) {
            const T e[6] = {f(k + 1), f(k), f(k - 1), f(k - 2), f(k - 3), f(k - 4)};
            wall_rhs<T, ORDER, true>(e, bd, hi_val, scale, q0, q1);
        }
    // ---- forward: rows 0, 1 and n-2, n-1 are not uniform rows and stay zero
    const Stencil<T, ORDER> S(scale);
    T y[MR], p = T(0);
#pragma unroll
    for (int k = 0; k < MR; k++) {
        T t = S(f(k - 2), f(k - 1), v[k], f(k + 1), f(k + 2)) - A * p;
        if (k < 2) t = G.j == 0 ? T(0) : t;
        y[k] = p = t;
    }
    // the carry out of a lane: its last row (lanes that hold row n-2 or follow it send nothing)
    const bool up = G.active && G.j < G.jn2;
    T Z = T(0);
#pragma unroll
    for (int i = 0; i < NT; i++) Z = from_prev(up ? y[MR - 1] + Q * Z : T(0));
    if constexpr (X::ON) Z += cut.carry_up(up ? y[MR - 1] + Q * Z : T(0));
    // (rows 0, 1 of the lower wall stay zero: lane 0 receives no carry)
#pragma unroll
    for (int k = 0; k < MR && k < uni_reach<T, ORDER>(); k++) y[k] += (T)uni_pow<ORDER>(k + 1) * Z;
    // ---- upper wall: row n-2 from y of row n-3, which starts the backward recurrence
    const bool dhi = bd == 1 || bd == 2, dlo = bd == 1 || bd == 3;
    // (needed where row n-2 may sit first in its lane)
    const T yprev = (REM < 0 || REM == 2) ? from_prev(y[MR - 1]) : T(0);
    T xn1 = T(0);
#pragma unroll
    for (int k = 0; k < MR; k++)
        if (k == kn2) {
            T xn2;
            upper_wall<T, ORDER>(k > 0 ? y[k > 0 ? k - 1 : 0] : yprev, q0, q1, dhi, xn2, xn1);
            y[k] = G.at_n2 ? xn2 : y[k];
        } else if (k > kn2) {
            y[k] = G.j >= G.jn2 ? T(0) : y[k];
        }
    if ((REM < 0 || REM == 1) && G.j > G.jn2) {
#pragma unroll
        for (int k = 0; k < MR; k++) y[k] = T(0);
    }
    // ---- backward
    T xp = T(0);
#pragma unroll
    for (int k = MR - 1; k >= 0; k--) {
        xp = y[k] - A * xp;
        x[k] = xp;
    }
    const bool dn = G.active && G.j > 0;
    const T xf = x[0];
    Z = T(0);
#pragma unroll
    for (int i = 0; i < NT; i++) Z = from_next(dn ? xf + Q * Z : T(0));
    if constexpr (X::ON) Z += cut.carry_down(dn ? xf + Q * Z : T(0));
#pragma unroll
    for (int k = MR - 1; k >= 0 && MR - k <= uni_reach<T, ORDER>(); k--) x[k] += (T)uni_pow<ORDER>(MR - k) * Z;
    // ---- lower wall: rows 0, 1 and the correction of the rows above, passed up the lanes
    T x0, x1;
    T c = lower_wall<T, ORDER>(x[2], r0, r1, dlo, x0, x1) * (T)uni_pow<ORDER>(-2);
    c = G.first ? c : T(0);
    T cs = c;
#pragma unroll
    for (int i = 1; i < NT; i++) {
        c = from_prev(up ? c : T(0)) * Q;
        cs += c;
    }
#pragma unroll
    for (int k = 0; k < MR; k++) x[k] += (T)uni_pow<ORDER>(k) * cs;
    x[0] = G.first ? x0 : x[0];
    x[1] = G.first ? x1 : x[1];
    return xn1;
}

// puts row n-1 (returned by line_solve on row n-2's lane) in its place
template <typename T, int MR, int REM>
__device__ __forceinline__ void line_last(const LineShape<MR, REM> &G, T xn1, T (&x)[MR]) {
#pragma unroll
    for (int k = 0; k < MR - 1; k++)
        if (k == G.kn2) x[k + 1] = G.at_n2 ? xn1 : x[k + 1];
    if (G.kn2 == MR - 1) {
        const T t = from_prev(G.at_n2 ? xn1 : T(0));
        x[0] = (G.active && G.j == G.jn2 + 1) ? t : x[0];
    }
}

}  // namespace cssx
