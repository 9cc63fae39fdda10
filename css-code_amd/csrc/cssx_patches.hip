// Batched compact derivatives of many independent patches of uneven shape in one launch
// (gfx950).  Each patch is a small subdomain f(nth, nphi, nr) with walls on all six
// faces (the Dbydr/Dbydt/Dbydp closures of derivatives.f90:547-796, :1010-1262 applied on
// every axis, as Determine_Dtype's dtype 0 would ask); all three first derivatives of every
// patch are work items of one kernel:
//   * r and phi items (seg_item): a workgroup of NT lanes covers P = NT/S columns cut into S segments (a power
//     of two) of M-4 .. M rows, lane = segment * P + column, the columns numbered over both pencil indices;
//   * theta items (line_item): every wavefront walks whole pencils in runs of MR rows per lane;
// both with the constant-coefficient recurrences of cssx_uniform.hpp: an item reads no plan, a seg_item
// exchanges its carries at two barriers and a line_item has none.  Pencils too short for them (fewer than
// 32 rows in FP32, 48 in FP64) run on the plan-driven strided_item / contig_item.
// One workgroup per item.  As many workgroups as are resident at once, each looping over the table, ran in step: all
// loading, then all storing; started one by one as others end they spread out.  16 patches of 32..512 points per
// axis in FP32: 3284 -> 2791 us (8 rows per lane of a theta item), 3238 -> 2494 (16 rows; 5.0 TB/s); sets of 8 to 12
// smaller ones 294 -> 277 and 289 -> 266, in FP64 621 -> 584 and 620 -> 553 (8 rows), 636 -> 610 and 615 -> 579 (16).
// (MR, NT) are template choices: start_variant picks the one a set starts with, and
// cssx_patchset_autotune times the instantiated variants on the actual patch set.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <map>
#include <new>
#include <tuple>
#include <vector>

#include "../../include/cssx.h"
#include "cssx_bufio.hpp"
#include "cssx_internal.hpp"
#include "cssx_kernels.hpp"
#include "cssx_line.hpp"
#include "cssx_plan.hpp"
#include "cssx_rows.hpp"

namespace cssx {

template <typename T>
struct PatchJob {
    const T *in;
    T *out;
    const T *plan;
    int n, na, nb, lanes;   // pencil length, pencils (a fast, b slow), SM or lanes per pencil
    long sa, sb, srow;
    T scale;
    int bdry, kind;         // 0 strided and 1 contiguous (plan-driven), 2 segments, 3 lines
    // kind 2: columns are na x nb flattened (nb = 1 where they lie back to back); S segments of base + 1 (the
    // first rem) or base rows, P = 2^lgp columns per item, and the powers of -a of those lengths
    int S, lgp, M, base, rem;
    T q0, q1, up0, up1;
};
enum PatchKind { PK_STRIDED = 0, PK_CONTIG = 1, PK_SEG = 2, PK_LINE = 3 };

constexpr int kPatchTail = 3 * kMaxLanes + 2 * kPcrSteps * kMaxLanes;
// capacity of each padded interface exchange array: SM*(P+1) or P*(SM+1) = NT + max(SM, P)
// slots with P = NT/SM, at most 2*NT
__host__ __device__ constexpr int patch_shared(int nt) { return 2 * nt; }

// A raw buffer resource over bytes [0, bytes) of base: loads outside it read zero and stores
// outside it are dropped (the range check of raw buffers), which replaces per-row bounds tests.
// A lane with no pencil takes the offset kNoPencil; a row below zero wraps to >= 2^32 - 4*rowb.
// The host keeps (n + 20) * rowb <= 2^31, so that neither can come back into range.
constexpr unsigned kNoPencil = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t span_rsrc(const void *base, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000);
}

// First-derivative right-hand side rows st .. st+MS-1 of a pencil of n rows with walls at
// both ends (prescribed wall derivatives zero): w[i] holds row st-4+i (zero outside the
// pencil) and end(k) returns row n-1-k.  Interior rows everywhere, then the wall closures in
// the segment that starts the pencil (rows 0, 1) and in the one or two that end it (rows
// n-2, n-1).
template <typename T, int MS, class End>
__device__ __forceinline__ void patch_rows(T (&d)[MS], const T *w, int st, int n, int bd, End end) {
#pragma unroll
    for (int jj = 0; jj < MS; jj++) d[jj] = Rows<T, 1>::interior(w[jj + 2], w[jj + 3], w[jj + 5], w[jj + 6]);
    if (st == 0) {
        const T r1 = Rows<T, 1>::wall1(w[4], w[5], w[6], w[7], w[8]);
        d[1] = r1;
        d[0] = Rows<T, 1>::wall0(bd == 1 || bd == 3, T(0), w[4], w[5], w[6], w[7], r1);
    }
    const int jl = n - 1 - st;   // row n-1 at jj = jl
    if (jl >= 0 && jl <= MS) {
        const T e0 = end(0), e1 = end(1), e2 = end(2), e3 = end(3), e4 = end(4);
        const T rn2 = -Rows<T, 1>::wall1(e0, e1, e2, e3, e4);
        const T rn1 = Rows<T, 1>::wall0(bd == 1 || bd == 2, T(0), e0, e1, e2, e3, -rn2);
        const T vn1 = (bd == 1 || bd == 2) ? -rn1 : rn1;
#pragma unroll
        for (int jj = 0; jj < MS; jj++) {
            if (jj == jl) d[jj] = vn1;
            if (jj == jl - 1) d[jj] = rn2;
        }
    }
}

template <typename T, int M, int NT>
__device__ __forceinline__ void strided_item(const PatchJob<T> &J, int ablk, int b, T *sp) {
    constexpr int W = M + 8;
    const int n = J.n, nl = (n + M - 1) / M, nI = nl - 1, SM = J.lanes, P = NT / SM;
    const int pn = n + nl;
    const int tid = threadIdx.x, lane = tid & 63;
    // exchange arrays with one padding slot per row ([segment][pencil] stride PS, [pencil]
    // [segment] stride XS), so that the lanes of a wavefront, which walk the other index, hit
    // different banks
    const int PS = P + 1, XS = SM + 1;
    constexpr int XC = patch_shared(NT);
    T *sh_xf = sp + 5 * pn, *sh_xl = sh_xf + XC, *sh_dI = sh_xl + XC, *sh_xI = sh_dI + XC;
    T *sh_tail = sh_xI + XC;
    const T *cf = sp, *cl = cf + pn, *cu = cl + pn, *vL = cu + pn, *vR = vL + pn;
    const int s = tid / P, p = tid - s * P;
    const long a = (long)ablk * P + p;
    const bool pen_ok = a < J.na, seg_ok = s < nl;
    const int st = s * M;
    const int m = seg_ok ? min(M, n - st) : 0;
    const long bofs = (long)b * J.sb;
    const unsigned rowb = (unsigned)J.srow * (unsigned)sizeof(T);
    // the resource spans rows [0, n) of the item's pencils: halo rows past the walls read zero
    // and stores of rows >= n, of lanes without a pencil or a segment, are dropped
    const unsigned lofs = pen_ok ? (unsigned)(a * J.sa) * (unsigned)sizeof(T) : kNoPencil;
    const unsigned span = (unsigned)n * rowb;
    const int sr = seg_ok ? st : n;
    const __amdgpu_buffer_rsrc_t rin = span_rsrc(J.in + bofs, span);
    const unsigned v0 = lofs + (unsigned)(sr - 4) * rowb;
    T w[W];
#pragma unroll
    for (int i = 0; i < W; i++) w[i] = bload<T>(rin, v0 + (unsigned)i * rowb, 0u);
    // plan staged in LDS while the rows are in flight: segment tables with one slot of padding
    // per segment, then the interface-solve tables
    for (int i = tid; i < 5 * n; i += NT) {
        const int c = i / n, r = i - c * n;
        sp[c * pn + r + r / M] = J.plan[i];
    }
    for (int i = tid; i < kPatchTail; i += NT) sh_tail[i] = J.plan[5 * n + i];
    T d[M];
    patch_rows<T, M>(d, w, sr, n, J.bdry, [&](int k) { return bload<T>(rin, lofs + (unsigned)(n - 1 - k) * rowb, 0u); });
    __syncthreads();   // plan staged
    const bool has_iface = seg_ok && s < nI;
    const int mi = has_iface ? M - 1 : m;
    const int pst = st + s;
    const T dI = d[M - 1];
    T y = T(0);
#pragma unroll
    for (int jj = 0; jj < M; jj++)
        if (jj < mi) {
            y = cf[pst + jj] * d[jj] - cl[pst + jj] * y;
            d[jj] = y;
        }
    T xn = T(0);
#pragma unroll
    for (int jj = M - 1; jj >= 0; jj--)
        if (jj < mi) {
            xn = d[jj] - cu[pst + jj] * xn;
            d[jj] = xn;
        }
    sh_xf[s * PS + p] = d[0];
    sh_xl[s * PS + p] = d[M - 2];
    sh_dI[s * PS + p] = dI;
    __syncthreads();
    {
        const int q = tid & (SM - 1), pp = tid / SM;
        const bool iq = q < nI && (long)ablk * P + pp < J.na;
        const T *rl = sh_tail, *ru = rl + kMaxLanes, *k1 = ru + kMaxLanes, *k2 = k1 + kPcrSteps * kMaxLanes,
                *invb = k2 + kPcrSteps * kMaxLanes;
        const int qc = q < kMaxLanes ? q : kMaxLanes - 1;
        T R = T(0);
        if (iq) R = sh_dI[q * PS + pp] - rl[qc] * sh_xl[q * PS + pp] - ru[qc] * sh_xf[(q + 1) * PS + pp];
        int steps = 0;
        while ((1 << steps) < nI) steps++;
        for (int k = 0; k < steps; k++) {
            const int dd = 1 << k;
            const T Rm = __shfl(R, lane - dd, 64);
            const T Rp = __shfl(R, lane + dd, 64);
            if (iq) R = R - k1[k * kMaxLanes + qc] * Rm - k2[k * kMaxLanes + qc] * Rp;
        }
        sh_xI[pp * XS + q] = iq ? R * invb[qc] : T(0);
    }
    __syncthreads();
    const T xl = (s > 0 && seg_ok) ? sh_xI[p * XS + s - 1] : T(0);
    const T xr = has_iface ? sh_xI[p * XS + s] : T(0);
    const __amdgpu_buffer_rsrc_t rout = span_rsrc(J.out + bofs, span);
    const unsigned o0 = lofs + (unsigned)sr * rowb;
#pragma unroll
    for (int jj = 0; jj < M; jj++) {
        const T x = (jj < mi) ? d[jj] + vL[pst + jj] * xl + vR[pst + jj] * xr : xr;
        bstore(J.scale * x, rout, o0 + (unsigned)jj * rowb, 0u);
    }
}

template <typename T, int MR, int NT>
__device__ __forceinline__ void contig_item(const PatchJob<T> &J, int ablk, int b, T *sp) {
    constexpr int W = MR + 8;
    const int n = J.n, nl = (n + MR - 1) / MR, nI = nl - 1, Lw = J.lanes, nT = nl * MR;
    const int tid = threadIdx.x, lane = tid & 63;
    const T *cf = sp, *cl = cf + nT, *cu = cl + nT, *vL = cu + nT, *vR = vL + nT;
    const T *rl = sp + 5 * nT, *ru = rl + kMaxLanes, *k1 = ru + kMaxLanes, *k2 = k1 + kPcrSteps * kMaxLanes,
            *invb = k2 + kPcrSteps * kMaxLanes;
    const int j = lane & (Lw - 1);
    const int ppw = 64 / Lw;
    const long a = ((long)ablk * (NT / 64) + (tid >> 6)) * ppw + lane / Lw;
    const bool pen_ok = a < J.na, active = pen_ok && j < nl;
    const int st = j * MR;
    const int m = active ? min(MR, n - st) : 0;
    // the resource spans the item's plane of pencils (contiguous rows, srow 1): a run's rows
    // past n belong to the next pencil and are zeroed below, lanes without a pencil read zero
    // and their stores are dropped
    const unsigned pofs = pen_ok ? (unsigned)(a * J.sa) * (unsigned)sizeof(T) : kNoPencil;
    const unsigned span = (unsigned)(J.na * J.sa) * (unsigned)sizeof(T);
    const __amdgpu_buffer_rsrc_t rin = span_rsrc(J.in + (long)b * J.sb, span);
    const unsigned o0 = pofs + (unsigned)st * (unsigned)sizeof(T);
    T v[MR];
#pragma unroll
    for (int k = 0; k < MR; k++) v[k] = bload<T>(rin, o0 + (unsigned)(k * sizeof(T)), 0u);
    // plan staged in LDS (row-major over runs, so lanes read consecutive slots) while the rows
    // are in flight
    for (int i = tid; i < 5 * n; i += NT) {
        const int c = i / n, r = i - c * n;
        const int jl = r / MR, jr = r - jl * MR;
        sp[c * nT + jr * nl + jl] = J.plan[i];
    }
    for (int i = tid; i < kPatchTail; i += NT) sp[5 * nT + i] = J.plan[5 * n + i];
#pragma unroll
    for (int k = 0; k < MR; k++)
        if (k >= m) v[k] = T(0);
    // halo rows from the neighbouring lanes by DPP wave shifts.  The first run's left halo
    // (rows < 0) and the last run's right halo (rows >= n) must read zero: the lanes that feed
    // them across a pencil boundary (the last lane of the previous pencil, the first lane of the
    // next) send zero, and inactive lanes hold zero runs.  The masking sits on the sending side
    // so that no select follows a shift: the compiler may turn such a select into an exec-masked
    // branch around the shift, whose source lanes then read as disabled (zero).
    T w[W];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        w[k] = from_prev(j == Lw - 1 ? T(0) : v[MR - 4 + k]);
        w[MR + 4 + k] = from_next(j == 0 ? T(0) : v[k]);
    }
#pragma unroll
    for (int k = 0; k < MR; k++) w[4 + k] = v[k];
    T d[MR];
    patch_rows<T, MR>(d, w, st, n, J.bdry,
                      [&](int k) { return bload<T>(rin, pofs + (unsigned)((n - 1 - k) * sizeof(T)), 0u); });
    __syncthreads();   // plan staged
    const bool has_iface = active && j < nI;
    const int mi = has_iface ? MR - 1 : m;
    const T dI = d[MR - 1];
    T y = T(0);
#pragma unroll
    for (int jj = 0; jj < MR; jj++)
        if (jj < mi) {
            y = cf[jj * nl + j] * d[jj] - cl[jj * nl + j] * y;
            d[jj] = y;
        }
    T xn = T(0);
#pragma unroll
    for (int jj = MR - 1; jj >= 0; jj--)
        if (jj < mi) {
            xn = d[jj] - cu[jj * nl + j] * xn;
            d[jj] = xn;
        }
    const T xf_next = __shfl(d[0], lane + 1, 64);
    T R = T(0);
    if (has_iface) R = dI - rl[j] * d[MR - 2] - ru[j] * xf_next;
    int steps = 0;
    while ((1 << steps) < nI) steps++;
    for (int s = 0; s < steps; s++) {
        const int dd = 1 << s;
        const T Rm = __shfl(R, lane - dd, 64);
        const T Rp = __shfl(R, lane + dd, 64);
        if (has_iface) R = R - k1[s * kMaxLanes + j] * Rm - k2[s * kMaxLanes + j] * Rp;
    }
    const T xI = has_iface ? R * invb[j] : T(0);
    T xl = __shfl(xI, lane - 1, 64);
    if (j == 0) xl = T(0);
    // rows past n (the next pencil's) go to an offset outside the resource
    const __amdgpu_buffer_rsrc_t rout = span_rsrc(J.out + (long)b * J.sb, span);
#pragma unroll
    for (int jj = 0; jj < MR; jj++) d[jj] = J.scale * ((jj < mi) ? d[jj] + vL[jj * nl + j] * xl + vR[jj * nl + j] * xI : xI);
    if (m == MR) {
        // a full run as 16-byte stores (buffer stores need 4-byte alignment only)
        constexpr int NC = MR * (int)sizeof(T) / 16;
#pragma unroll
        for (int c = 0; c < NC; c++) {
            cssx_u32x4 q;
            __builtin_memcpy(&q, &d[c * (16 / (int)sizeof(T))], 16);
            __builtin_amdgcn_raw_buffer_store_b128(q, rout, o0 + (unsigned)(c * 16), 0u, 0);
        }
    } else {
#pragma unroll
        for (int jj = 0; jj < MR; jj++) bstore(d[jj], rout, jj < m ? o0 + (unsigned)(jj * sizeof(T)) : kNoPencil, 0u);
    }
}

// S segments of the columns [blk*P, +P) (the recurrences and exchanges of k_deriv_seg)
template <typename T, int M, int NT>
__device__ __forceinline__ void seg_item(const PatchJob<T> &J, int blk, T *sp) {
    using U = Uni<1>;
    constexpr int TAIL = 5, REACH = uni_reach<T, 1>(), NTERM = (REACH + M - TAIL) / (M - TAIL + 1);
    constexpr T a_ = (T)U::a;
    T *sh_y = sp, *sh_x = sp + NT, *sh_lo = sp + 2 * NT;   // sh_lo: two values per column
    const int tid = threadIdx.x, n = J.n, S = J.S, P = 1 << J.lgp;
    const int k = tid >> J.lgp, p = tid & (P - 1);
    const int st = k * J.base + min(k, J.rem), m = J.base + (k < J.rem ? 1 : 0);
    const bool lo = k == 0, hi = k == S - 1;
    const unsigned cols = (unsigned)J.na * (unsigned)J.nb, c = (unsigned)blk * P + p;
    unsigned a = c, b = 0;
    if (J.nb > 1) {
        b = c / (unsigned)J.na;
        a = c - b * (unsigned)J.na;
    }
    const unsigned rowb = (unsigned)J.srow * (unsigned)sizeof(T);
    // the resource spans the patch: loads of lanes without a column read zero, their stores are dropped
    const unsigned span = (unsigned)n * (unsigned)J.na * (unsigned)J.nb * (unsigned)sizeof(T);
    const unsigned lofs = c < cols ? (a * (unsigned)J.sa + b * (unsigned)J.sb) * (unsigned)sizeof(T) : kNoPencil;
    const __amdgpu_buffer_rsrc_t rin = span_rsrc(J.in, span);
    // w[i] = row st - 2 + i; past a wall any row of the pencil will do
    T w[M + 4];
    const unsigned v0 = lofs + (unsigned)st * rowb;
    {
        const int dlo = lo ? 2 : 0;
#pragma unroll
        for (int i = 0; i < M + 4; i++) {
            if (i < 2) w[i] = bload<T>(rin, lofs + (unsigned)(st - 2 + i + dlo) * rowb, 0u);
            else if (i >= M - TAIL + 3) w[i] = bload<T>(rin, lofs + (unsigned)min(st - 2 + i, n - 1) * rowb, 0u);
            else w[i] = bload<T>(rin, v0, (unsigned)(i - 2) * rowb);
        }
    }
    const T scale = J.scale;
    const int bd = J.bdry;
    T r0 = T(0), r1 = T(0), q0 = T(0), q1 = T(0);
    if (lo) {
        const T e[6] = {w[2], w[3], w[4], w[5], w[6], w[7]};
        wall_rhs<T, 1, false>(e, bd, T(0), scale, r0, r1);
    }
    if (hi) {
        T e[6];   // row n-1 sits at w[m + 1]
#pragma unroll
        for (int t = 0; t < 6; t++) {
            e[t] = w[M + 1 - t];
#pragma unroll
            for (int s = 1; s < TAIL; s++) e[t] = m == M - s ? w[M + 1 - t - s] : e[t];
        }
        wall_rhs<T, 1, true>(e, bd, T(0), scale, q0, q1);
    }
    const Stencil<T, 1> St(scale);
    const int me = hi ? m - 2 : m;
    T y[M], yp = T(0), yl = T(0);
#pragma unroll
    for (int j = 0; j < M; j++) {
        T t = St(w[j], w[j + 1], w[j + 2], w[j + 3], w[j + 4]) - a_ * yp;
        if (j < 2) t = lo ? T(0) : t;
        if (j > M - TAIL - 3) t = j < me ? t : T(0);
        y[j] = yp = t;
        if (j >= M - TAIL - 2) yl = j < me ? t : yl;
    }
    sh_y[tid] = yl;
    __syncthreads();
    auto qseg = [&](int s) -> T { return s < J.rem ? J.q1 : J.q0; };
    T Y = T(0);
#pragma unroll
    for (int t = NTERM; t >= 1; t--)
        if (k - t >= 0) Y = sh_y[(k - t) * P + p] + qseg(k - t) * Y;
#pragma unroll
    for (int j = 0; j < M && j < REACH + 2; j++) {
        const T t = y[j] + (T)uni_pow<1>(j + 1) * Y;
        y[j] = j > M - TAIL - 3 ? (j < me ? t : y[j]) : t;
    }
    T xn1 = T(0);
    if (hi) {
        T y3 = y[M - 3], xn2;
#pragma unroll
        for (int s = 1; s < TAIL; s++) y3 = m == M - s ? y[M - 3 - s] : y3;
        upper_wall<T, 1>(y3, q0, q1, bd == 1 || bd == 2, xn2, xn1);
#pragma unroll
        for (int s = 0; s < TAIL; s++) y[M - 2 - s] = m == M - s ? xn2 : y[M - 2 - s];
    }
    T xp = T(0);
#pragma unroll
    for (int j = M - 1; j >= 0; j--) {
        xp = y[j] - a_ * xp;
        y[j] = xp;
    }
    sh_x[tid] = y[0];
    if (lo) {
        sh_lo[p] = y[2];
        sh_lo[P + p] = r1 - (T)U::l1 * r0;
    }
    __syncthreads();
    auto carry_x = [&](int kk) -> T {
        T X = T(0);
#pragma unroll
        for (int t = NTERM; t >= 1; t--)
            if (kk + t < S) X = sh_x[(kk + t) * P + p] + qseg(kk + t) * X;
        return X;
    };
    {
        const T X = carry_x(k) * (k < J.rem ? J.up1 : J.up0);
#pragma unroll
        for (int j = M - 1; j >= 0 && M - j <= REACH + TAIL; j--) y[j] += (T)uni_pow<1>(M - j) * X;
    }
    T x0 = T(0), x1 = T(0);
    if (k <= (NTERM == 1 ? 0 : NTERM)) {
        const T x2 = sh_lo[p] + (T)uni_pow<1>(-2) * (qseg(0) * carry_x(0));
        T s = lower_wall<T, 1>(x2, T(0), sh_lo[P + p], bd == 1 || bd == 3, x0, x1) * (T)uni_pow<1>(-2);
        if constexpr (NTERM > 1) {
            T f = T(1);
            for (int t = 0; t < k; t++) f *= qseg(t);
            s *= f;
        }
#pragma unroll
        for (int j = 0; j < M && j < REACH + 2; j++) y[j] += (T)uni_pow<1>(j) * s;
        if (lo) {
            y[0] = x0 + r0;
            y[1] = x1;
        }
    }
    if (hi) {
#pragma unroll
        for (int s = 0; s < TAIL; s++) y[M - 1 - s] = m == M - s ? xn1 : y[M - 1 - s];
    }
    const __amdgpu_buffer_rsrc_t rout = span_rsrc(J.out, span);
#pragma unroll
    for (int j = 0; j < M; j++)
        if (j < M - TAIL + 1 || j < m) bstore(y[j], rout, v0, (unsigned)j * rowb);
}

// whole theta pencils [blk * pencils per workgroup, ...): every wavefront on its own
template <typename T, int MR, int NT>
__device__ __forceinline__ void line_item(const PatchJob<T> &J, int blk) {
    const int n = J.n, nl = J.lanes, ppw = 64 / nl;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int pl = (int)((unsigned)lane * (unsigned)J.lgp >> 16), j = lane - pl * nl;   // lgp: ceil(2^16 / nl)
    const unsigned np = (unsigned)J.na * (unsigned)J.nb, id0 = ((unsigned)blk * (NT / 64) + wv) * ppw;
    if (id0 >= np) return;
    const bool active = pl < ppw && id0 + pl < np;
    const long at0 = (long)id0 * n, total = (long)np * n - at0;
    const unsigned at = active ? (unsigned)(pl * n + j * MR) : 0u;
    LineShape<MR, -1> G(n, nl, j, active);
    T v[MR], x[MR];
    line_load<T, MR>(J.in + at0, at, total, G, v);
    const T xn1 = line_solve<T, 1, MR>(G, v, J.bdry, T(0), T(0), J.scale, x);
    line_last<T, MR>(G, xn1, x);
    if (active) line_store<T, MR>(J.out + at0, at, G, x);
}

// FP32 is held to 64 VGPRs: eight waves per SIMD (two 1024-lane or four 512-lane workgroups per CU)
template <typename T, int MR, int NT>
__global__ __launch_bounds__(NT, (sizeof(T) == 4 && MR == 8) ? 8 : 1) void k_patch_derivs(const PatchJob<T> *__restrict__ jobs,
                                                       const int4 *__restrict__ items) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T *sp = reinterpret_cast<T *>(smem_raw);
    const int4 w = items[xcd_neighbour(blockIdx.x, gridDim.x)];
    const PatchJob<T> &J = jobs[w.x];
    if (J.kind == PK_LINE) {
        line_item<T, MR, NT>(J, w.y);
    } else if (J.kind == PK_SEG) {
        if constexpr (sizeof(T) == 4) {
            switch (J.M) {
            case 20: seg_item<T, 20, NT>(J, w.y, sp); break;
            case 24: seg_item<T, 24, NT>(J, w.y, sp); break;
            case 28: seg_item<T, 28, NT>(J, w.y, sp); break;
            default: seg_item<T, 32, NT>(J, w.y, sp); break;
            }
        } else {
            if (J.M == 12) seg_item<T, 12, NT>(J, w.y, sp);
            else seg_item<T, 16, NT>(J, w.y, sp);
        }
    } else if (J.kind == PK_STRIDED) {
        strided_item<T, 16, NT>(J, w.y, w.z, sp);
    } else {
        contig_item<T, 8, NT>(J, w.y, w.z, sp);
    }
}

// rows from which a patch axis runs on the constant-coefficient items
template <typename T>
constexpr int patch_uniform_min() { return sizeof(T) == 4 ? 32 : 48; }

// LDS bytes: the exchange arrays of a seg_item, and the plan-driven items' for their longest pencil
inline size_t patch_lds(int nmax_short, int NT, size_t elem) {
    const size_t seg = (size_t)4 * NT;
    if (nmax_short == 0) return seg * elem;
    const int nl = (nmax_short + 15) / 16;
    const size_t a = (size_t)5 * (nmax_short + nl) + 4 * (size_t)patch_shared(NT) + kPatchTail;
    const size_t b = (size_t)5 * 8 * ((nmax_short + 7) / 8) + kPatchTail;
    return std::max({seg, a, b}) * elem;
}

// the variants the autotuner chooses from: rows per lane of the theta items and workgroup size
constexpr int kPatchVariants = 4;
constexpr int kVarMR[kPatchVariants] = {8, 8, 16, 16};
constexpr int kVarNT[kPatchVariants] = {1024, 512, 1024, 512};

// ---- synthetic patch data: N(0,1) (SplitMix64 + Box-Muller, the generator of cssx/model.py's
//      normal()) smoothed by [1,2,1]/4 along each axis with the edge value repeated --------------
__device__ __forceinline__ double splitmix_u01(unsigned long long seed, unsigned long long idx) {
    unsigned long long z = seed * 0x9E3779B97F4A7C15ull + idx * 0x9E3779B97F4A7C15ull + 0x632BE59BD9B4E5B5ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z = z ^ (z >> 31);
    return ((double)(z >> 11) + 0.5) * (1.0 / 9007199254740992.0);
}

template <typename T>
__global__ __launch_bounds__(256) void k_patch_noise(T *out, long n, unsigned long long seed) {
    const long i = item_index();
    if (i >= n) return;
    const long m = (n + 1) / 2, k = i >> 1;
    const double u1 = splitmix_u01(seed, (unsigned long long)k), u2 = splitmix_u01(seed, (unsigned long long)(m + k));
    const double rad = sqrt(-2.0 * log(u1));
    const double ang = 6.283185307179586476925286766559 * u2;
    out[i] = (T)((i & 1) ? rad * sin(ang) : rad * cos(ang));
}

// out = [1,2,1]/4 of in along one axis (element stride `stride`, length len), edges repeated
template <typename T>
__global__ __launch_bounds__(256) void k_patch_smooth(const T *__restrict__ in, T *__restrict__ out, long n, long stride,
                                                      int len) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int q = (int)((i / stride) % len);
    const T c = in[i];
    const T lo = q > 0 ? in[i - stride] : c;
    const T hi = q < len - 1 ? in[i + stride] : c;
    out[i] = T(0.25) * (lo + hi) + T(0.5) * c;
}

}  // namespace cssx

using namespace cssx;

extern "C" int cssx_normal_fill(void *out, int prec, long n, unsigned long long seed, void *stream) {
    if (!out || n < 1 || (prec != CSSX_PREC_F64 && prec != CSSX_PREC_F32)) return CSSX_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    if (prec == CSSX_PREC_F64)
        hipLaunchKernelGGL(k_patch_noise<double>, item_grid(n), dim3(256), 0, s, (double *)out, n, seed);
    else
        hipLaunchKernelGGL(k_patch_noise<float>, item_grid(n), dim3(256), 0, s, (float *)out, n, seed);
    return hipGetLastError() == hipSuccess ? CSSX_OK : CSSX_EHIP;
}

extern "C" int cssx_patch_fill(void *out, void *tmp, int prec, int nr, int nth, int nphi, unsigned long long seed,
                               void *stream) {
    if (!out || !tmp || nr < 1 || nth < 1 || nphi < 1 || (prec != CSSX_PREC_F64 && prec != CSSX_PREC_F32))
        return CSSX_EINVAL;
    const long n = (long)nr * nth * nphi;
    const unsigned g = (unsigned)((n + 255) / 256);
    hipStream_t s = (hipStream_t)stream;
    if (prec == CSSX_PREC_F64) {
        double *o = (double *)out, *t = (double *)tmp;
        hipLaunchKernelGGL(k_patch_noise<double>, item_grid(n), dim3(256), 0, s, t, n, seed);
        hipLaunchKernelGGL(k_patch_smooth<double>, dim3(g), dim3(256), 0, s, t, o, n, 1L, nth);
        hipLaunchKernelGGL(k_patch_smooth<double>, dim3(g), dim3(256), 0, s, o, t, n, (long)nth, nphi);
        hipLaunchKernelGGL(k_patch_smooth<double>, dim3(g), dim3(256), 0, s, t, o, n, (long)nth * nphi, nr);
    } else {
        float *o = (float *)out, *t = (float *)tmp;
        hipLaunchKernelGGL(k_patch_noise<float>, item_grid(n), dim3(256), 0, s, t, n, seed);
        hipLaunchKernelGGL(k_patch_smooth<float>, dim3(g), dim3(256), 0, s, t, o, n, 1L, nth);
        hipLaunchKernelGGL(k_patch_smooth<float>, dim3(g), dim3(256), 0, s, o, t, n, (long)nth, nphi);
        hipLaunchKernelGGL(k_patch_smooth<float>, dim3(g), dim3(256), 0, s, t, o, n, (long)nth * nphi, nr);
    }
    return hipGetLastError() == hipSuccess ? CSSX_OK : CSSX_EHIP;
}

struct cssx_patchset {
    int prec = 0, npatch = 0, nmax_short = 0, best = 0;   // nmax_short: longest plan-driven pencil
    long nitems[kPatchVariants] = {}, nplan[kPatchVariants] = {};   // items; the plan-driven ones among them
    void *jobs[kPatchVariants] = {};
    int4 *items[kPatchVariants] = {};
};

namespace {

unsigned next_pow2(unsigned v) {
    unsigned p = 1;
    while (p < v) p <<= 1;
    return p;
}

template <typename T>
int build_variant(cssx_patchset *ps, const cssx_patch *pt, int var) {
    const int MR = kVarMR[var], NT = kVarNT[var];
    std::vector<PatchJob<T>> jobs;
    std::vector<int4> items;
    const int prec = sizeof(T) == 8 ? CSSX_PREC_F64 : CSSX_PREC_F32;
    auto pw = [](int k) {
        double v = 1.0;
        for (int i = 0; i < std::abs(k); i++) v *= -Uni<1>::a;
        return (T)(k < 0 ? 1.0 / v : v);
    };
    for (int i = 0; i < ps->npatch; i++) {
        const cssx_patch &q = pt[i];
        const long sth = 1, sph = q.nth, sr = (long)q.nth * q.nphi;
        void *outs[3] = {q.d_r, q.d_th, q.d_ph};
        for (int ax = 0; ax < 3; ax++) {
            if (!outs[ax]) continue;
            PatchJob<T> J{};
            J.in = (const T *)q.in;
            J.out = (T *)outs[ax];
            J.bdry = q.bdry;
            if (ax == 0) { J.n = q.nr; J.na = q.nth; J.nb = q.nphi; J.sa = sth; J.sb = sph; J.srow = sr; J.scale = (T)q.dri; }
            else if (ax == 1) { J.n = q.nth; J.na = q.nphi; J.nb = q.nr; J.sa = sph; J.sb = sr; J.srow = sth; J.scale = (T)q.dti; }
            else { J.n = q.nphi; J.na = q.nth; J.nb = q.nr; J.sa = sth; J.sb = sr; J.srow = sph; J.scale = (T)q.dpi; }
            const bool uniform = J.n >= patch_uniform_min<T>();
            J.kind = ax == 1 ? (uniform ? PK_LINE : PK_CONTIG) : (uniform ? PK_SEG : PK_STRIDED);
            // the kernels' buffer ranges (span_rsrc): offsets up to kNoPencil + (n + 20) rows
            // stay below 2^32, and contiguous items walk unit-stride rows
            if (ax != 1 && (double)(J.n + 20) * (double)J.srow * sizeof(T) > 2147483648.0) return CSSX_EINVAL;
            if (ax == 1 && (J.srow != 1 || (double)J.na * (double)J.sa * sizeof(T) > 2147483648.0)) return CSSX_EINVAL;
            long per_b;
            int nb = J.nb;
            if (J.kind == PK_SEG) {
                // 32-row (FP32) or 16-row (FP64) segments at most, a power of two of them (a patch is at
                // most 2^30 bytes: the resource of its columns fits)
                const int most = sizeof(T) == 4 ? 32 : 16;
                J.S = (int)next_pow2((unsigned)((J.n + most - 1) / most));
                J.base = J.n / J.S;
                J.rem = J.n % J.S;
                J.M = (J.base + (J.rem > 0) + 3) / 4 * 4;
                J.lgp = 0;
                while ((J.S << (J.lgp + 1)) <= NT) J.lgp++;
                J.q0 = pw(J.base); J.q1 = pw(J.base + 1);
                J.up0 = pw(J.base - J.M); J.up1 = pw(J.base + 1 - J.M);
                if (J.sb == J.na) {   // r: the two pencil indices are one contiguous run
                    J.na *= J.nb;
                    J.nb = 1;
                }
                nb = 1;
                per_b = ((long)J.na * J.nb + (1 << J.lgp) - 1) >> J.lgp;
            } else if (J.kind == PK_LINE) {
                J.lanes = (J.n + MR - 1) / MR;
                J.lgp = (65536 + J.lanes - 1) / J.lanes;
                nb = 1;
                const long pw_ = (long)(NT / 64) * (64 / J.lanes);
                per_b = ((long)J.na * J.nb + pw_ - 1) / pw_;
            } else {
                PlanKey key{J.n, 1, END_WALL, END_WALL, q.bdry};
                key.variant = J.kind == PK_CONTIG ? 1 : 2;
                key.seg = J.kind == PK_CONTIG ? 8 : 16;
                const void *plan = nullptr;
                int rc = get_plan(key, prec, &plan);
                if (rc) return rc;
                J.plan = (const T *)plan;
                J.lanes = (int)next_pow2((unsigned)((J.n + key.seg - 1) / key.seg));
                const long p = J.kind == PK_CONTIG ? (long)(NT / 64) * (64 / J.lanes) : NT / J.lanes;
                per_b = (J.na + p - 1) / p;
                ps->nmax_short = std::max(ps->nmax_short, J.n);
                ps->nplan[var] += per_b * nb;
            }
            const int jid = (int)jobs.size();
            jobs.push_back(J);
            for (int b = 0; b < nb; b++)
                for (long x = 0; x < per_b; x++) items.push_back(make_int4(jid, (int)x, b, 0));
        }
    }
    if (items.size() > (size_t)INT32_MAX) return CSSX_EINVAL;
    ps->nitems[var] = (long)items.size();
    if (hipMalloc(&ps->jobs[var], std::max<size_t>(1, jobs.size()) * sizeof(PatchJob<T>)) != hipSuccess ||
        hipMalloc((void **)&ps->items[var], std::max<size_t>(1, items.size()) * sizeof(int4)) != hipSuccess)
        return CSSX_ENOMEM;
    if ((jobs.size() && hipMemcpy(ps->jobs[var], jobs.data(), jobs.size() * sizeof(PatchJob<T>), hipMemcpyHostToDevice) != hipSuccess) ||
        (items.size() && hipMemcpy(ps->items[var], items.data(), items.size() * sizeof(int4),
                                   hipMemcpyHostToDevice) != hipSuccess))
        return CSSX_EHIP;
    return CSSX_OK;
}

// The variant a set starts with.  1024 lanes to a workgroup, and the faster run length of each type (above); 512 lanes
// where more than three quarters of the items are plan-driven: those cover the pencils of one plane each and leave
// most of a large workgroup idle.  1024 -> 512 lanes (8 rows per lane) in FP32 / FP64: 256 patches of 16^3 169 -> 69 / 328 -> 133
// us, 64 of 8..31 points per axis 45 -> 23 / 101 -> 41, 60 of 8x8x512 294 -> 154 / 743 -> 304 (plan-driven items
// only), 300 of 32..64 719 -> 425 (FP64, 79% of the items), 4 of 500x20x500 96 -> 93 (FP32, 76%); with fewer it is the other
// way round: 4 of 500x20x500 218 -> 226 (FP64, 61%), 4 of 20x500x500 90 -> 93 / 211 -> 217 (52% / 35%), 24 of
// 32..256 324 -> 353 / 692 -> 737 (0 / 1%).
int start_variant(const cssx_patchset *ps) {
    const int v = ps->prec == CSSX_PREC_F32 ? 2 : 0;
    return 4 * ps->nplan[v] > 3 * ps->nitems[v] ? 1 : v;
}

template <typename T, int MR, int NT>
hipError_t launch_variant(const cssx_patchset *ps, int var, hipStream_t s) {
    const size_t shm = patch_lds(ps->nmax_short, NT, sizeof(T));
    const void *fn = (const void *)k_patch_derivs<T, MR, NT>;
    if (shm > 65536) {
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
        if (e != hipSuccess) return e;
    }
    // A launch counts its work-items in 32 bits, and one of more starts without an error but short of what the count
    // wraps by: a set of 2^22 items at 1024 lanes to a workgroup, or 2^23 at 512, takes more than one.
    const long n = ps->nitems[var], most = 0xffffffffL / NT;
    for (long at = 0; at < n; at += most) {
        hipLaunchKernelGGL((k_patch_derivs<T, MR, NT>), dim3((unsigned)std::min(most, n - at)), dim3(NT), shm, s,
                           (const PatchJob<T> *)ps->jobs[var], (const int4 *)ps->items[var] + at);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <typename T>
hipError_t launch_any(const cssx_patchset *ps, int var, hipStream_t s) {
    switch (var) {
    case 0: return launch_variant<T, 8, 1024>(ps, var, s);
    case 1: return launch_variant<T, 8, 512>(ps, var, s);
    case 2: return launch_variant<T, 16, 1024>(ps, var, s);
    default: return launch_variant<T, 16, 512>(ps, var, s);
    }
}

}  // namespace

extern "C" void cssx_patchset_destroy(cssx_patchset *ps) {
    if (!ps) return;
    (void)hipDeviceSynchronize();
    for (int v = 0; v < kPatchVariants; v++) {
        if (ps->jobs[v]) (void)hipFree(ps->jobs[v]);
        if (ps->items[v]) (void)hipFree(ps->items[v]);
    }
    delete ps;
}

extern "C" int cssx_patchset_create(const cssx_patch *patches, int npatch, int prec, cssx_patchset **out) {
    if (!patches || npatch < 1 || !out || (prec != CSSX_PREC_F64 && prec != CSSX_PREC_F32)) return CSSX_EINVAL;
    *out = nullptr;
    for (int i = 0; i < npatch; i++) {
        const cssx_patch &q = patches[i];
        if (!q.in || q.nr < 8 || q.nth < 8 || q.nphi < 8 || q.nr > 512 || q.nth > 512 || q.nphi > 512 || q.bdry < 0 ||
            q.bdry > 4)
            return CSSX_EINVAL;
        const double bytes = (double)q.nr * q.nth * q.nphi * (prec == CSSX_PREC_F64 ? 8.0 : 4.0);
        if (bytes >= 4294967295.0) return CSSX_EINVAL;   // 32-bit buffer offsets
    }
    cssx_patchset *ps = new (std::nothrow) cssx_patchset;
    if (!ps) return CSSX_ENOMEM;
    ps->prec = prec;
    ps->npatch = npatch;
    for (int v = 0; v < kPatchVariants; v++) {
        int rc = prec == CSSX_PREC_F64 ? build_variant<double>(ps, patches, v) : build_variant<float>(ps, patches, v);
        if (rc) {
            cssx_patchset_destroy(ps);
            return rc;
        }
    }
    ps->best = start_variant(ps);
    *out = ps;
    return CSSX_OK;
}

extern "C" int cssx_patchset_run(cssx_patchset *ps, int variant, void *stream) {
    if (!ps || variant < -1 || variant >= kPatchVariants) return CSSX_EINVAL;
    const int v = variant < 0 ? ps->best : variant;
    hipStream_t s = (hipStream_t)stream;
    hipError_t e = ps->prec == CSSX_PREC_F64 ? launch_any<double>(ps, v, s) : launch_any<float>(ps, v, s);
    return e == hipSuccess ? CSSX_OK : CSSX_EHIP;
}

extern "C" int cssx_patchset_autotune(cssx_patchset *ps, int reps, void *stream, int *best, float *ms_out) {
    if (!ps || reps < 1) return CSSX_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) return CSSX_EHIP;
    float bestms = 0.0f;
    int bv = 0;
    int rc = CSSX_OK;
    for (int v = 0; v < kPatchVariants && !rc; v++) {
        if ((rc = cssx_patchset_run(ps, v, stream))) break;   // warm
        if (hipEventRecord(e0, s) != hipSuccess) { rc = CSSX_EHIP; break; }
        for (int r = 0; r < reps && !rc; r++) rc = cssx_patchset_run(ps, v, stream);
        float ms = 0.0f;
        if (rc || hipEventRecord(e1, s) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
            hipEventElapsedTime(&ms, e0, e1) != hipSuccess) {
            rc = rc ? rc : CSSX_EHIP;
            break;
        }
        ms /= reps;
        if (ms_out) ms_out[v] = ms;
        if (v == 0 || ms < bestms) {
            bestms = ms;
            bv = v;
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc) return rc;
    ps->best = bv;
    if (best) *best = bv;
    return CSSX_OK;
}
