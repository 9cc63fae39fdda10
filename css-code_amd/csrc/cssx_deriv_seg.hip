// Compact derivative along a strided axis (r or phi) for gfx950, solved with the constant-coefficient
// recurrences of cssx_uniform.hpp: the operators of derivatives.f90 Dbydr / Dbydp (:547-796,
// :1480-1591) and D2bydr2 / D2bydp2 (:799-1007, :1594-1684) on walls at both ends or the periodic wrap.
//
// A pencil is cut into S balanced segments of m or m-1 rows (M-4 < m <= M).  A wavefront holds G
// segments of P = 64/G neighbouring columns (lane = g*P + p), so every row is one coalesced access of
// P values; the columns of a block are numbered over both pencil indices, so that a ragged theta length
// leaves no idle lanes.  Every lane loads its rows plus two on each side, runs the two recurrences in
// registers and exchanges two carries per segment through LDS (two barriers); no coefficients are read.
// Bound by HBM: one read and one write per point, the halo rows come from L2.  At 256x512x1024 in FP32 the
// r sweep takes 218 us and the phi sweep 223 (4.9 and 4.8 TB/s; a bare copy in the same access pattern 198 and
// 207) against 250 and 294 with plan coefficients and a reduced interface system; on a ragged 90x151x250
// grid 32 against 59-89 us for the fields of one right-hand side.  (One column per lane marching up the whole
// pencil, with no exchange at all, measured 216 and 212 us there but 46 against 32 us at 128x256x512.)
#include <hip/hip_runtime.h>

#include <algorithm>

#include "cssx_bufio.hpp"
#include "cssx_plan.hpp"
#include "cssx_uniform.hpp"

namespace cssx {

// host-computed powers of -a that depend on the launch's segment lengths
template <typename T>
struct SegArgs {
    int S, base, rem;      // segments; rows of a segment: base + 1 in the first rem, base in the others
    T q0, q1;              // (-a)^base, (-a)^(base+1)
    T up0, up1;            // (-a)^(base-M), (-a)^(base+1-M)
    int near_xcd;          // neighbouring columns on one XCD (xcd_neighbour)
};

// EVEN: every segment has M rows (n = S*M), which takes the tests on a segment's last rows out.
template <typename T, int ORDER, int M, int G, bool EVEN>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(G == 1 ? 8 : 1))) void k_deriv_seg(const DerivLaunch<T> L, const SegArgs<T> A) {
    using U = Uni<ORDER>;
    constexpr int P = 64 / G, TAIL = EVEN ? 1 : 4, REACH = uni_reach<T, ORDER>();
    constexpr int NT = (REACH + M - TAIL) / (M - TAIL + 1);   // segments a carry spans
    constexpr T a_ = (T)U::a;
    // (sh_end: what the end segments know of their closure rows, kept here instead of in registers)
    __shared__ T sh_y[1024], sh_x[1024], sh_lo[2][64], sh_end[4][64];
    const DerivJob<T> &J = L.jobs[blockIdx.y];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int p = lane & (P - 1);
    const int k = G == 1 ? wv : wv * G + lane / P;      // this lane's segment
    const int n = L.n, S = A.S;
    const bool seg_ok = k < S;
    // (lanes past the last segment read rows 0 .. of the pencil)
    const int st = seg_ok ? (EVEN ? k * M : k * A.base + min(k, A.rem)) : 2;
    const int m = EVEN ? M : seg_ok ? A.base + (k < A.rem ? 1 : 0) : 0;
    const bool lo = k == 0, hi = k == S - 1;
    // wave-uniform: whether the wavefront holds an end of the pencils (or segments past it)
    const bool edge = wv == 0 || (wv + 1) * G >= S;
    const bool wall = J.lo_kind == END_WALL;             // both ends, or the periodic wrap
    // column c of the launch: pencil (a, b); addresses relative to the block's first b
    const unsigned cols = (unsigned)L.na * (unsigned)L.nb, c0 = (A.near_xcd ? xcd_neighbour(blockIdx.x, gridDim.x) : blockIdx.x) * P;
    const bool pen_ok = c0 + p < cols;
    const bool active = pen_ok && seg_ok;
    unsigned a = c0 + (pen_ok ? p : 0), b = 0, b0 = 0;
    if (L.nb > 1) {
        b0 = c0 / (unsigned)L.na;
        b = a / (unsigned)L.na;
        a -= b * (unsigned)L.na;
    }
    const unsigned rowb = (unsigned)L.srow * (unsigned)sizeof(T);
    const unsigned lofs = (a * (unsigned)L.sa + (b - b0) * (unsigned)L.sb) * (unsigned)sizeof(T);
    const __amdgpu_buffer_rsrc_t rin = field_rsrc(J.in + (long)b0 * L.sb);
    const long gbase = (long)a * J.g_a + (long)b * J.g_b;
    // One workgroup of 16 wavefronts per CU: with two (64 registers) a full-size phi sweep moved its
    // 128-byte rows at 4.4 TB/s instead of 4.8.
    if constexpr (G == 2 && sizeof(T) == 4) asm volatile("" ::: "v71");
    // ---- 1. window: w[i] = row st - 2 + i.  Rows below 0 and from n on wrap on a periodic pencil; at a
    //         wall any row will do, as no uniform row reads them.
    T w[M + 4];
    const int dlo = lo ? (wall ? 2 : n) : 0, dhi = hi ? (wall ? TAIL + 2 : n) : 0;
    auto row_of = [&](int i) {   // i constant
        int q = st - 2 + i;
        if (i < 2) q += dlo;
        if (i >= M - TAIL + 3) q -= q >= n ? dhi : 0;
        return q;
    };
    const unsigned v0 = lofs + (unsigned)st * rowb;
#pragma unroll
    for (int i = 0; i < M + 4; i++) {
        if (G == 1) w[i] = bload<T>(rin, lofs, (unsigned)row_of(i) * rowb);
        else if (i < 2 || i >= M - TAIL + 3) w[i] = bload<T>(rin, lofs + (unsigned)row_of(i) * rowb, 0u);
        else w[i] = bload<T>(rin, v0, (unsigned)(i - 2) * rowb);
    }
    if (J.pre) {
#pragma unroll
        for (int i = 0; i < M + 4; i++) {
            w[i] *= J.pre[row_of(i)];
            if (G > 1 && i % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // few profile values in flight
        }
    }
    // ---- 2. wall and seam rows
    const T scale = J.scale;
    const int bd = J.bdry;
    T r0 = T(0), r1 = T(0), q0 = T(0), q1 = T(0);
    if (!edge) {
    } else if (wall) {
        if (lo) {
            const T val = (pen_ok && J.glo) ? J.glo[gbase] * J.neu_mul : T(0);
            const T e[6] = {w[2], w[3], w[4], w[5], w[6], w[7]};
            wall_rhs<T, ORDER, false>(e, bd, val, scale, r0, r1);
        }
        if (hi) {
            const T val = (pen_ok && J.ghi) ? J.ghi[gbase] * J.neu_mul : T(0);
            // row n-1 sits at w[m + 1]
            T e[6];
#pragma unroll
            for (int t = 0; t < 6; t++) {
                e[t] = w[M + 1 - t];
#pragma unroll
                for (int s = 1; s < TAIL; s++) e[t] = m == M - s ? w[M + 1 - t - s] : e[t];
            }
            wall_rhs<T, ORDER, true>(e, bd, val, scale, q0, q1);
        }
    } else {
        // periodic: the seam rows take the neighbour's derivative from the explicit formula
        if (lo) {
            T g0, g1;   // rows -4, -3
            g0 = bload<T>(rin, lofs + (unsigned)(n - 4) * rowb, 0u);
            g1 = bload<T>(rin, lofs + (unsigned)(n - 3) * rowb, 0u);
            if (J.pre) {
                g0 *= J.pre[n - 4];
                g1 *= J.pre[n - 3];
            }
            if constexpr (ORDER == 1) r0 = Rows<T, 1>::halo_lo0(g0, g1, w[0], w[1], w[2], w[3], w[4], T(1));
            else r0 = Rows<T, 2>::halo_lo0(g0, g1, w[0], w[1], w[2], w[3], w[4]);
        }
        if (hi) {
            T g2 = bload<T>(rin, lofs + 2u * rowb, 0u), g3 = bload<T>(rin, lofs + 3u * rowb, 0u);
            if (J.pre) {
                g2 *= J.pre[2];
                g3 *= J.pre[3];
            }
            T e[5];   // rows n-3, n-2, n-1, and 0, 1
#pragma unroll
            for (int t = 0; t < 5; t++) {
                e[t] = w[M - 1 + t];
#pragma unroll
                for (int s = 1; s < TAIL; s++) e[t] = m == M - s ? w[M - 1 + t - s] : e[t];
            }
            if constexpr (ORDER == 1) q0 = Rows<T, 1>::halo_hi0(e[0], e[1], e[2], e[3], e[4], g2, g3, T(1));
            else q0 = Rows<T, 2>::halo_hi0(e[0], e[1], e[2], e[3], e[4], g2, g3);
        }
    }
    if (edge) {
        if (lo) {
            sh_end[0][p] = wall ? r0 : (T)((double)scale * (1.0 / U::p)) * r0;
            sh_end[1][p] = r1;
        }
        if (hi) {
            sh_end[2][p] = wall ? q0 : (T)((double)scale * (1.0 / U::p)) * q0;
            sh_end[3][p] = q1;
        }
    }
    // ---- 3. forward recurrence; rows >= me are not uniform rows of this segment and stay zero
    const Stencil<T, ORDER> St(scale);
    const int me = (wall && hi) ? m - 2 : m;
    T y[M], yp = T(0), yl = T(0);
#pragma unroll
    for (int j = 0; j < M; j++) {
        T d = St(w[j], w[j + 1], w[j + 2], w[j + 3], w[j + 4]);
        if (j == 0 && edge) d = (lo && !wall) ? sh_end[0][p] : d;
        if (j > M - TAIL - 1 && edge) d = (hi && !wall && j == m - 1) ? sh_end[2][p] : d;
        T t = d - a_ * yp;
        if (j < 2) t = (lo && wall) ? T(0) : t;
        if (j > M - TAIL - 3) t = j < me ? t : T(0);
        y[j] = yp = t;
        if (j >= M - TAIL - 2) yl = j < me ? t : yl;
    }
    sh_y[wv * 64 + lane] = yl;
    __syncthreads();
    // carry-in from the segments below: Y = yl_{k-1} + (-a)^{m_{k-1}} (yl_{k-2} + ...)
    auto qseg = [&](int s) -> T { return EVEN ? (T)uni_pow<ORDER>(M) : s < A.rem ? A.q1 : A.q0; };
    T Y = T(0);
#pragma unroll
    for (int t = NT; t >= 1; t--) {
        const int s = k - t;
        if (s >= 0 && seg_ok) Y = sh_y[s * P + p] + qseg(s) * Y;
    }
    // Y's weight in y_j falls below the rounding after REACH rows
    const T Yw = Y;
#pragma unroll
    for (int j = 0; j < M && j < REACH + 2; j++) {
        const T t = y[j] + (T)uni_pow<ORDER>(j + 1) * Yw;
        y[j] = j > M - TAIL - 3 ? (j < me ? t : y[j]) : t;
    }
    // ---- upper wall: row n-2 starts the backward recurrence
    if (wall && hi) {
        T xn1;
        T y3 = y[M - 3], xn2;
#pragma unroll
        for (int s = 1; s < TAIL; s++) y3 = m == M - s ? y[M - 3 - s] : y3;
        upper_wall<T, ORDER>(y3, sh_end[2][p], sh_end[3][p], bd == 1 || bd == 2, xn2, xn1);
#pragma unroll
        for (int s = 0; s < TAIL; s++)
            if (m == M - s) y[M - 2 - s] = xn2;
        sh_end[2][p] = xn1;
    }
    // ---- 4. backward recurrence
    T xp = T(0);
#pragma unroll
    for (int j = M - 1; j >= 0; j--) {
        xp = y[j] - a_ * xp;
        y[j] = xp;
    }
    sh_x[wv * 64 + lane] = y[0];
    if (lo) {
        if (wall) {
            sh_lo[0][p] = y[2];
            sh_lo[1][p] = sh_end[1][p] - (T)U::l1 * sh_end[0][p];
        } else {
            sh_lo[0][p] = y[0];
        }
    }
    __syncthreads();
    // carry-in from the segments above: X = xf_{k+1} + (-a)^{m_{k+1}} (xf_{k+2} + ...)
    auto carry_x = [&](int kk) -> T {
        T X = T(0);
#pragma unroll
        for (int t = NT; t >= 1; t--) {
            const int s = kk + t;
            if (s < S) X = sh_x[s * P + p] + qseg(s) * X;
        }
        return X;
    };
    {
        const T X = EVEN ? carry_x(k) : seg_ok ? carry_x(k) * (k < A.rem ? A.up1 : A.up0) : T(0);
#pragma unroll
        for (int j = M - 1; j >= 0 && M - j <= REACH + TAIL; j--) y[j] += (T)uni_pow<ORDER>(M - j) * X;
    }
    // ---- 5. lower end: the correction s (-a)^(row - 2) (wall) or s (-a)^row (periodic)
    T x0 = T(0), x1 = T(0);
    if (NT == 1 ? lo : k <= NT) {
        // every segment it reaches forms s from segment 0's numbers
        T s;
        if (wall) {
            const T x2 = sh_lo[0][p] + (T)uni_pow<ORDER>(-2) * (qseg(0) * carry_x(0));
            s = lower_wall<T, ORDER>(x2, T(0), sh_lo[1][p], bd == 1 || bd == 3, x0, x1) * (T)uni_pow<ORDER>(-2);
            // (x0 came out without its own right-hand side, which only segment 0 holds)
            if (lo) x0 += sh_end[0][p];
        } else {
            s = (T)(-U::a * U::a) * (sh_lo[0][p] + qseg(0) * carry_x(0));
        }
        if constexpr (NT > 1) {
            // times (-a)^st
            T f = T(1);
            for (int t = 0; t < k; t++) f *= qseg(t);
            s *= f;
        }
#pragma unroll
        for (int j = 0; j < M && j < REACH + 2; j++) y[j] += (T)uni_pow<ORDER>(j) * s;
        if (wall && lo) {
            y[0] = x0;
            y[1] = x1;
        }
    }
    if (wall && hi) {
#pragma unroll
        for (int s = 0; s < TAIL; s++)
            if (m == M - s) y[M - 1 - s] = sh_end[2][p];
    }
    // ---- 6. store
    if (!active) return;
    const bool has_pm = J.mul_a || J.mul_b;
    const T pm = (J.mul_a ? J.mul_a[a] : T(1)) * (J.mul_b ? J.mul_b[b] : T(1));
    const T beta = J.beta;
    const T *__restrict__ post = J.post;
    const __amdgpu_buffer_rsrc_t rout = field_rsrc(J.out + (long)b0 * L.sb);
    auto ofs = [&](int j, unsigned &v, unsigned &s) {
        v = G == 1 ? lofs : v0;
        s = G == 1 ? (unsigned)(st + j) * rowb : (unsigned)j * rowb;
    };
    // with beta != 0 the old values of four rows are loaded ahead of their stores (a store may
    // alias the next row's load, so a load per store would wait a memory round trip each)
    constexpr int C = 4;
#pragma unroll
    for (int jc = 0; jc < M; jc += C) {
        if (G > 1) __builtin_amdgcn_sched_barrier(0);
        T old[C];
#pragma unroll
        for (int t = 0; t < C; t++) {
            unsigned v, s;
            ofs(jc + t, v, s);
            old[t] = (beta != T(0) && jc + t < m) ? bload<T>(rout, v, s) : T(0);
        }
#pragma unroll
        for (int t = 0; t < C; t++) {
            const int j = jc + t;
            if (j < M - TAIL + 1 || j < m) {
                unsigned v, s;
                ofs(j, v, s);
                T o = y[j];
                if (post) o *= post[st + j];
                if (has_pm) o *= pm;
                if (beta != T(0)) o += beta * old[t];
                bstore(o, rout, v, s);
            }
        }
    }
}

// (M, G, S) of a pencil of n rows: S segments whose lengths ceil(n/S) and floor(n/S) both lie in
// (M-4, M] of an instantiated M, G per wavefront.  Segments of up to 32 (FP32) / 16 (FP64) rows, the
// most a lane holds without spilling, re-read the fewest halo rows and serve fields that come from memory;
// for fields that stay in the L2s shorter chains end sooner.  FP32, one field, 32- against 16- against
// 8-row segments: 128x256x512 27.0, 30.7, 33.2 us; 97x203x331 (26 MB) 16.6, 18.3, 20.9; 90x151x250 (14 MB) 10.8,
// 9.4, 11.9; right-hand side of 64x64x128 points (2 MB a field, up to 6 a launch) 113, 101, 97; FP64 there 139
// (16) and 135 (8).  False if n has none.
bool seg_shape(int n, bool f64, long cols, int njobs, int &M, int &G, int &S) {
    const double mb = (double)n * (double)cols * (f64 ? 8.0 : 4.0) / 1e6;
    const int want = njobs > 1 && mb <= 4.5 ? 8 : f64 || mb <= 16.0 ? 16 : 32;
    bool found = false;
    for (int most = f64 ? 16 : 32; most >= 8; most /= 2) {
        const int g = n <= 16 * most ? 1 : n <= 32 * most ? 2 : 4;
        if (found && g > 1) break;
        if (n > 16 * g * most || (!f64 && g > 2)) break;
        const int least = g == 1 ? 8 : f64 ? 12 : 20;
        for (int s = (n + most - 1) / most; s <= 16 * g; s++) {
            const int m = ((n + s - 1) / s + 3) / 4 * 4;
            if (m < least) break;
            if (n / s > m - 4) {
                found = true;
                M = m;
                G = g;
                S = s;
                break;
            }
        }
        if (found && most <= want) break;
    }
    return found;
}

// Whether a lane's rows lie within 32-bit byte offsets of its block's first slow index.  A block's up to 64 columns run
// over the end of the fast index: t slow indices on, its last lane is at fast index na + 62 - t * na at most.
bool seg_span_fits(int n, int na, int nb, long sa, long sb, long srow, size_t elem) {
    double span = 0.0;
    for (int t = 0; t < nb && (long)t * na <= na + 62L; t++) {
        const long a = t == 0 ? na - 1L : std::min(na - 1L, na + 62L - (long)t * na);
        span = std::max(span, (double)t * (double)sb + (double)a * (double)sa);
    }
    return (span + (double)(n - 1) * (double)srow + 1.0) * (double)elem < 4294967295.0;
}

template <typename T>
hipError_t launch_deriv_seg(const DerivLaunch<T> &L0, int order, hipStream_t stream) {
    DerivLaunch<T> L = L0;
    int M, G, S;
    if (!seg_shape(L.n, sizeof(T) == 8, (long)L.na * L.nb, L.njobs, M, G, S) || L.njobs < 1 || L.njobs > kMaxJobs || L.n < 32)
        return hipErrorInvalidValue;
    const int P = 64 / G;
    bool flat = L.nb > 1 && L.sa == 1 && L.sb == L.na;
    for (int i = 0; i < L.njobs; i++) {
        const DerivJob<T> &J = L.jobs[i];
        flat = flat && !J.mul_a && !J.mul_b && ((!J.glo && !J.ghi) || J.g_b == J.g_a * L.na);
    }
    // (a field past the 32-bit offsets keeps its slow index in the base pointer)
    flat = flat && ((double)L.na * L.nb + (double)(L.n - 1) * L.srow) * sizeof(T) < 4294967295.0;
    if (!flat && !seg_span_fits(L.n, L.na, L.nb, L.sa, L.sb, L.srow, sizeof(T))) return hipErrorInvalidValue;
    if (flat) {   // the two pencil indices are one contiguous run
        L.na = L.na * L.nb;
        L.nb = 1;
    }
    const double a = order == 1 ? Uni<1>::a : Uni<2>::a;
    auto pw = [&](int k) {
        double v = 1.0;
        for (int i = 0; i < (k < 0 ? -k : k); i++) v *= -a;
        return (T)(k < 0 ? 1.0 / v : v);
    };
    SegArgs<T> A;
    A.S = S;
    A.base = L.n / S;
    A.rem = L.n % S;
    A.q0 = pw(A.base);
    A.q1 = pw(A.base + 1);
    A.up0 = pw(A.base - M);
    A.up1 = pw(A.base + 1 - M);
    const long cols = (long)L.na * L.nb;
    const dim3 grid((unsigned)((cols + P - 1) / P), L.njobs), block(64 * ((S + G - 1) / G));
    const bool even = L.n == S * M;
    // Neighbouring columns on one XCD: in launches of more workgroups than the chip holds several times over
    // (256x512x1024 FP32 phi 224 -> 201 us, r 217 -> 215; ragged 311x333x411 r 109 -> 90), and on phi also in
    // smaller ones whose rows are no whole lines (97x203x331 20.6 -> 18.7).  Small r sweeps, whose rows lie
    // whole planes apart, lost by it (97x203x331 16.6 -> 19.5).
    const bool lines = ((long)L.na * sizeof(T)) % 128 == 0;
    A.near_xcd = grid.x > 2048 || (L.nb > 1 && !lines);
#define CSSX_LAUNCH_S(MM, GG)                                                                                     \
    do {                                                                                                          \
        if (even) {                                                                                               \
            if (order == 1) hipLaunchKernelGGL((k_deriv_seg<T, 1, MM, GG, true>), grid, block, 0, stream, L, A);  \
            else hipLaunchKernelGGL((k_deriv_seg<T, 2, MM, GG, true>), grid, block, 0, stream, L, A);             \
        } else {                                                                                                  \
            if (order == 1) hipLaunchKernelGGL((k_deriv_seg<T, 1, MM, GG, false>), grid, block, 0, stream, L, A); \
            else hipLaunchKernelGGL((k_deriv_seg<T, 2, MM, GG, false>), grid, block, 0, stream, L, A);            \
        }                                                                                                         \
        return hipGetLastError();                                                                                 \
    } while (0)
    if constexpr (sizeof(T) == 4) {
        if (G == 1) {
            switch (M) {
            case 8: CSSX_LAUNCH_S(8, 1);
            case 12: CSSX_LAUNCH_S(12, 1);
            case 16: CSSX_LAUNCH_S(16, 1);
            case 20: CSSX_LAUNCH_S(20, 1);
            case 24: CSSX_LAUNCH_S(24, 1);
            case 28: CSSX_LAUNCH_S(28, 1);
            case 32: CSSX_LAUNCH_S(32, 1);
            }
        } else if (G == 2) {
            switch (M) {
            case 20: CSSX_LAUNCH_S(20, 2);
            case 24: CSSX_LAUNCH_S(24, 2);
            case 28: CSSX_LAUNCH_S(28, 2);
            case 32: CSSX_LAUNCH_S(32, 2);
            }
        }
    } else {
        if (G == 1) {
            switch (M) {
            case 8: CSSX_LAUNCH_S(8, 1);
            case 12: CSSX_LAUNCH_S(12, 1);
            case 16: CSSX_LAUNCH_S(16, 1);
            }
        } else if (G == 2) {
            switch (M) {
            case 12: CSSX_LAUNCH_S(12, 2);
            case 16: CSSX_LAUNCH_S(16, 2);
            }
        } else {
            switch (M) {
            case 12: CSSX_LAUNCH_S(12, 4);
            case 16: CSSX_LAUNCH_S(16, 4);
            }
        }
    }
#undef CSSX_LAUNCH_S
    return hipErrorInvalidValue;
}

template hipError_t launch_deriv_seg<float>(const DerivLaunch<float> &, int, hipStream_t);
template hipError_t launch_deriv_seg<double>(const DerivLaunch<double> &, int, hipStream_t);

}  // namespace cssx
