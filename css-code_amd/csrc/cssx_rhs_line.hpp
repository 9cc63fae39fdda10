// Every pointwise term of the right-hand side together with the theta derivatives it needs (gfx950).
// Included by cssx_rhs.hip.
//
// The lanes of a workgroup hold whole theta pencils, MR = 4 consecutive points each, so the seven theta
// derivatives are solved where they are used (line_solve: registers and DPP shifts; a pencil cut by the end
// of a wavefront passes its carries through LDS) instead of being written by sweeps and read back, and
// the theta-wall density closure reads the momentum tendency of the end points from the lanes that hold
// them.  The terms are those of main_terms and final_point, in their order, over the lane's points.
//
// Bound by memory: per stage the seven theta sweeps' 14 fields of traffic and the final kernel's 7
// reads of them go away.  256x512x1024 FP32 RK4 stage: 6.95 ms of k_rhs_final + 1.30 of theta sweeps
// + 0.1 of k_walls_gather -> 6.00 ms, now 5.68 (average of the four stages); 128x256x512 FP64:
// 1.63 + 0.42 -> 1.43, now 1.36.  Eight points per lane (512 rows in one wavefront, one wavefront per
// SIMD) took 8.53 ms, three wavefronts per SIMD (spills) 10.3 ms.
#pragma once

#include "cssx_line.hpp"

namespace cssx {

// boundary codes and wall values of the theta derivatives (w v u s bp br rho)
template <typename T>
struct LineTheta {
    int bw, bv, bu, bs, bbp, bbr, brho;
    const T *tv_lo, *tv_hi, *tbp_lo, *tbp_hi;   // by pencil (ir * nphi + ip)
    const T *rr_lo, *rr_hi;                     // the density's radial wall derivatives in x-space (nphi, nth)
    T scale, neu;
    // The strip: the workgroup's lanes from `off` on hold `pencils` pencils of nl lanes each; inv_nl = ceil(2^16 / nl)
    unsigned inv_nl;
    int nl, pencils, off;
    int near_xcd;   // neighbouring workgroups on one XCD (xcd_neighbour)
};

// k / w for w = 3 or 6 (rw = 1/w), rounded as the division is: the remainder of k rw is exact, and adding its
// quotient rounds correctly; div_fixup passes zeros, infinities and NaN as the division does
__device__ __forceinline__ float div_by(float k, float w, float rw) {
    const float q = k * rw;
    return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-q, w, k), rw, q), w, k);
}
__device__ __forceinline__ double div_by(double k, double w, double rw) {
    const double q = k * rw;
    return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-q, w, k), rw, q), w, k);
}

// MR values `at` values after p, which must lie in p[0, total) unless CHK (then those past the end are
// zero).  p is the same for the workgroup: a scalar base and a 32-bit lane offset.
template <typename T, int MR, bool CHK>
__device__ __forceinline__ void run_load(const T *__restrict__ p, unsigned at, long total, T (&v)[MR]) {
    if (!CHK || (long)at + MR <= total) {
        __builtin_memcpy(v, (const char *)p + at * (unsigned)sizeof(T), sizeof(v));
    } else {
#pragma unroll
        for (int k = 0; k < MR; k++) v[k] = (long)at + k < total ? p[at + k] : T(0);
    }
}

// Bound of field iv (bound_value) over the lane's points
template <typename T, int MR, int REM>
__device__ __forceinline__ void bound_run(int iv, const LineShape<MR, REM> &G, int it0, int ir, T (&v)[MR], const BoundFlags &f,
                                          int nr, const T *sr1) {
    const bool bot = ir == 0, top = ir == nr - 1, mag = f.magnetic && iv >= 5;
    const bool ends = iv == 1 || (iv == 3 && !f.theta_stress_free) || (mag && (f.perf_cond ? iv != 5 : iv == 5));
    const bool all = iv == 3 ? bot || top
                     : iv == 1 || iv == 2 ? (bot && !f.bot_sf) || (top && !f.top_sf)
                                          : iv == 7 && mag && ((bot && f.bot_radial) || (top && f.top_radial));
    if (iv == 4 && f.bot_ctemp && bot) {
#pragma unroll
        for (int k = 0; k < MR; k++) v[k] = sr1[min(it0 + k, G.n - 1)];
    }
#pragma unroll
    for (int k = 0; k < MR; k++)
        v[k] = (all || (ends && ((k == 0 && G.first) || (k == G.m - 1 && G.last)))) ? T(0) : v[k];
}

// One RK4 stage (stage_value) of all NV fields over the lane's points, ST = 1, 2 (stages 2 and 3) or 4.  Everything
// it reads is asked for before the first value is written: field by field, each would wait for memory
// behind the stores of the one before (256x512x1024 FP32: 7.08 -> 6.00 ms a stage).
template <typename T, int MR, int NV, int ST, bool CHK>
struct StageRun {
    static constexpr bool F64 = sizeof(T) == 8;
    using Y = std::conditional_t<F64 || ST == 4, double, float>;
    Y y[NV][MR];      // y0 (FP32 stages 1 to 3: its FP32 copy)
    T s[NV][MR];      // stage 1: the SLD tendency; else the running sum
    __device__ __forceinline__ void load(const StageFuse<T> &F, long N, long base, unsigned at) {
        const long left = N - base;
#pragma unroll
        for (int iv = 0; iv < NV; iv++) {
            const long o = iv * N + base;
            if constexpr (std::is_same<Y, double>::value) run_load<double, MR, CHK>(F.y0 + o, at, left, y[iv]);
            else run_load<float, MR, CHK>((const float *)F.y0f + o, at, left, y[iv]);
            if constexpr (ST == 1) {
                if (F.dif) run_load<T, MR, CHK>(F.dif + o, at, left, s[iv]);
            } else if constexpr (F64) {
                run_load<T, MR, CHK>((const T *)F.acc64 + o, at, left, s[iv]);
            } else {
                run_load<T, MR, CHK>((const T *)F.acc32 + o, at, left, s[iv]);
            }
        }
    }
    // k: the tendency of field iv
    template <int REM>
    __device__ __forceinline__ void finish(const StageFuse<T> &F, const Consts<T> &c, const LineShape<MR, REM> &G, int iv, long base,
                                           unsigned at, int it0, int ir, const T (&k)[MR]) {
        const long o = (long)iv * c.N + base;
        constexpr T w = ST == 2 ? T(3) : T(6), rw = T(1) / w;
#pragma unroll
        for (int q = 0; q < MR; q++) {
            if constexpr (ST == 1) s[iv][q] = F.dif ? s[iv][q] + div_by(k[q], w, rw) : k[q];
            else s[iv][q] = s[iv][q] + div_by(k[q], w, rw);
        }
        if constexpr (ST != 4) {
            if constexpr (F64) line_store<T, MR>((T *)F.acc64 + o, at, G, s[iv]);
            else line_store<T, MR>((T *)F.acc32 + o, at, G, s[iv]);
            const T h = (T)(F.stage == 3 ? F.dt : 0.5 * F.dt);
#pragma unroll
            for (int q = 0; q < MR; q++) y[iv][q] = y[iv][q] + h * k[q];
            bound_run(iv, G, it0, ir, y[iv], F.f, c.nr, (const T *)F.sr1_t);
            line_store<T, MR>((T *)F.y1 + o, at, G, y[iv]);
        } else {
#pragma unroll
            for (int q = 0; q < MR; q++) y[iv][q] = y[iv][q] + F.dt * (double)s[iv][q];
            bound_run(iv, G, it0, ir, y[iv], F.f, c.nr, F.sr1_64);
            line_store<double, MR>(F.y0 + o, at, G, y[iv]);
            if (!F64 && !F.last) {
                const double bg = iv == 0 ? F.rbar64[ir] : iv == 4 ? F.sbar64[ir] : 0.0;
#pragma unroll
                for (int q = 0; q < MR; q++) s[iv][q] = (T)(y[iv][q] - bg);
                line_store<T, MR>(F.y0f + o, at, G, s[iv]);
            }
        }
    }
};

template <typename T, int MR, int REM, bool MAG, bool CUT, bool CHK>
__device__ __forceinline__ void rhs_line(const Consts<T> &c, const Prof<T> &P, const T *st, const T *B, const T *dr_rho, T *dv,
                                         const StageFuse<T> &F, const float *__restrict__ ext, const T *D,
                                         const LineTheta<T> &H, LineCut<T, 7, 4> &cutmem) {
    constexpr int NT = (uni_reach<T, 1>() + MR - 1) / MR;
    const int n = c.nth, nl = H.nl;
    const int lane = threadIdx.x & 63, s0 = (int)threadIdx.x - H.off;
    const int pl = s0 < 0 ? H.pencils : (int)((unsigned)s0 * H.inv_nl >> 16);
    constexpr bool FL = sizeof(T) == 4;   // fluctuation form (Consts::fluct)
    unsigned bx = blockIdx.x;
    int ir = (int)blockIdx.y;
    if (H.near_xcd) {   // (the last workgroup stays the last)
        const unsigned i = xcd_neighbour(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
        ir = (int)(i / gridDim.x);
        bx = i - (unsigned)ir * gridDim.x;
    }
    const unsigned ip0 = bx * (unsigned)H.pencils;
    const unsigned id0 = (unsigned)ir * (unsigned)c.nphi + ip0;
    const bool active = pl < H.pencils && ip0 + pl < (unsigned)c.nphi;
    // lanes without a pencil work along on the first one and store nothing
    const unsigned id = active ? id0 + pl : id0;
    const int j = active ? s0 - pl * nl : 0;
    const int it0 = j * MR;
    const long N = c.N, base = (long)id0 * n;   // the workgroup's first point
    const unsigned at = active ? (unsigned)(pl * n + it0) : 0u;
    const LineShape<MR, REM> G(n, nl, j, active);
    LineAcross<T, MR, 7, 4> cut{cutmem, 0, __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane, false, false, T(0), T(0)};
    if constexpr (CUT) {
        // rows from the cut: a pencil's lanes below and above it lie side by side
        cut.from_below = active && lane < NT && j > lane;
        cut.from_above = active && 63 - lane < NT && nl - 1 - j > 63 - lane;
        T q = T(1), qs = T(0), qb = T(0);
#pragma unroll
        for (int i = 0; i < NT; i++) {
            qs = lane == i ? q : qs;
            qb = 63 - lane == i ? q : qb;
            q *= (T)uni_pow<1>(MR);
        }
        cut.q_below = qs;
        cut.q_above = qb;
    }
#define CSSX_K _Pragma("unroll") for (int k = 0; k < MR; k++)
    auto field = [&](const T *p, T(&v)[MR]) { run_load<T, MR, CHK>(p + base, at, N - base, v); };
    auto slot = [&](int s, T(&v)[MR]) { run_load<T, MR, CHK>(D + ((long)s * N + base), at, N - base, v); };
    auto theta = [&](const T *p, T(&v)[MR]) {
        if constexpr (REM == 0) {
            run_load<T, MR, false>(p, it0, n, v);
        } else {
            CSSX_K v[k] = p[min(it0 + k, n - 1)];
        }
    };
    // theta derivative of f with the prescribed wall derivatives wl, wh (f keeps its rows)
    auto dth = [&](int fld, const T(&f)[MR], int bd, T wl, T wh, T(&x)[MR]) {
        T v[MR], xn1;
        CSSX_K v[k] = f[k];
        if constexpr (CUT) {
            cut.f = fld;
            xn1 = line_solve<T, 1, MR>(G, v, bd, wl * H.neu, wh * H.neu, H.scale, x, cut);
        } else {
            xn1 = line_solve<T, 1, MR>(G, v, bd, wl * H.neu, wh * H.neu, H.scale, x);
        }
        line_last<T, MR>(G, xn1, x);
    };
    // A workgroup stays within one radius, whose profiles are scalars, and everything small is asked for here: loads
    // return in order, so one in the middle of the terms waits for whatever is in flight before it.  RK4 step,
    // against workgroups across radii that read the profiles where they use them: 256x512x1024 FP32 52.6 -> 50.3 ms,
    // 128x256x512 FP64 12.3 -> 11.9, 90x151x250 FP32 (two steps) 3.85 -> 3.61, 48x96x96 FP32 RHS 77.2 -> 74.0 us.
    const T ri = P.rinv[ir], rv = P.r[ir], epsr = P.eps[ir], g0 = FL ? P.hres[ir] : -P.grav[ir];
    const T rb = FL ? P.rbar[ir] : T(0), tbar = FL ? P.tbar[ir] : T(0), dsb = FL ? P.dsbar[ir] : T(0);
    const T tr = FL ? P.tr[ir] : T(0), drb = FL ? P.drbar[ir] : T(0);
    const T erl = P.erl[ir], erh = P.erh[ir];
    const T omsq = rv * c.omega0 * c.omega0, om2 = c.om2;
    T cot[MR], sn[MR], cs[MR], csc[MR];
    theta(P.cot, cot);
    theta(P.sn, sn);
    theta(P.cs, cs);
    theta(P.csc, csc);
    const T vl = (G.first && H.tv_lo) ? H.tv_lo[id] : T(0), vh = (G.at_n2 && H.tv_hi) ? H.tv_hi[id] : T(0);
    const T bl = (MAG && G.first && H.tbp_lo) ? H.tbp_lo[id] : T(0), bh = (MAG && G.at_n2 && H.tbp_hi) ? H.tbp_hi[id] : T(0);
    T W[MR], V[MR], U[MR], rs[MR], Bt[MR], Bp[MR], Br[MR], S[MR];
    field(st, rs);
    field(st + 4 * N, S);
    field(st + N, W);
    field(st + 2 * N, V);
    field(st + 3 * N, U);
    if constexpr (MAG) {
        field(B, Bt);
        field(B + N, Bp);
        field(B + 2 * N, Br);
    }
    if constexpr (CUT) {
        cut.post(0, W);
        cut.post(1, V);
        cut.post(2, U);
        cut.post(3, S);
        if constexpr (MAG) {
            cut.post(4, Bp);
            cut.post(5, Br);
        }
        cut.post(6, rs);
        cut.barrier();
    }
    T Rho[MR], t[MR], ta[MR], tb[MR];
    CSSX_K {
        const Thermo<T> th = thermo_at<T, FL>(rs[k], S[k], rb, tbar, c);
        Rho[k] = th.rho;
        t[k] = th.t;
        ta[k] = th.a;
        tb[k] = th.b;
    }
    T xdw[MR], xdv[MR], xdu[MR], xdrho[MR], xds[MR], x[MR];
    // ---- Source_Theta_Terms (rhs_mpi.f90:812-1027)
    {
        dth(0, W, H.bw, T(0), T(0), x);
        CSSX_K {
            xdw[k] = omsq * sn[k] * cs[k];
            xdu[k] = g0 + omsq * sn[k] * sn[k];
            xdrho[k] = -Rho[k] * W[k] * cot[k] * ri;
            xdv[k] = -om2 * cs[k] * W[k];
            xdu[k] = xdu[k] + ri * W[k] * W[k];
            const T wk = x[k] * ri;
            xdrho[k] = xdrho[k] - Rho[k] * wk;
            xdw[k] = xdw[k] - W[k] * wk;
            xdw[k] = xdw[k] + V[k] * (ri * cot[k] * V[k] + om2 * cs[k]);
            xdv[k] = xdv[k] - ri * V[k] * W[k] * cot[k];
            xdu[k] = xdu[k] + V[k] * (ri * V[k] + om2 * sn[k]);
        }
        dth(1, V, H.bv, vl, vh, x);
        CSSX_K {
            xdv[k] = xdv[k] - W[k] * (x[k] * ri);
            xdrho[k] = xdrho[k] - T(2) * ri * Rho[k] * U[k];
            xdv[k] = xdv[k] - U[k] * (ri * V[k] + om2 * sn[k]);
            xdw[k] = xdw[k] - ri * U[k] * W[k];
        }
    }
    dth(2, U, H.bu, T(0), T(0), x);
    CSSX_K xdu[k] = xdu[k] - W[k] * (x[k] * ri);
    dth(3, S, H.bs, T(0), T(0), x);
    CSSX_K {
        const T wk = x[k] * ri;
        xds[k] = (fabs(epsr) > T(0)) ? epsr * (T(1) / Rho[k]) / t[k] : T(0);
        xdw[k] = xdw[k] - c.gamm1 * t[k] * wk;
        xds[k] = xds[k] - W[k] * wk;
    }
    if constexpr (MAG) {
        dth(4, Bp, H.bbp, bl, bh, x);
        CSSX_K {
            const T oorho = (T(1) / Rho[k]) * T(kOneOver4Pi) * ri;
            xdu[k] = xdu[k] - Bt[k] * Bt[k] * oorho;
            xdw[k] = xdw[k] - Bp[k] * Bp[k] * cot[k] * oorho;
            xdv[k] = xdv[k] + Bp[k] * Bt[k] * cot[k] * oorho;
            xdu[k] = xdu[k] - Bp[k] * Bp[k] * oorho;
            const T wk = x[k] * oorho;
            xdv[k] = xdv[k] + Bt[k] * wk;
            xdw[k] = xdw[k] - Bp[k] * wk;
        }
        dth(5, Br, H.bbr, T(0), T(0), x);
        CSSX_K {
            const T oorho = (T(1) / Rho[k]) * T(kOneOver4Pi) * ri;
            const T wk = x[k] * oorho;
            xdw[k] = xdw[k] + Br[k] * (Bt[k] * oorho - wk);
            xdv[k] = xdv[k] + Br[k] * Bp[k] * oorho;
            xdu[k] = xdu[k] + Bt[k] * wk;
        }
    }
    // ---- Phi_Terms (rhs_mpi.f90:1064-1260)
    {
        T oors[MR];
        CSSX_K oors[k] = ri * csc[k];
        slot(D_PRHO, x);
        CSSX_K {
            const T wk = x[k] * oors[k];
            xdrho[k] = xdrho[k] - V[k] * wk;
            xdv[k] = xdv[k] - c.pconst * wk * t[k] * (T(1) / Rho[k]);
        }
        slot(D_PV, x);
        CSSX_K {
            const T wk = x[k] * oors[k];
            xdv[k] = xdv[k] - V[k] * wk;
            xdrho[k] = xdrho[k] - Rho[k] * wk;
        }
        slot(D_PW, x);
        CSSX_K xdw[k] = xdw[k] - V[k] * (x[k] * oors[k]);
        slot(D_PU, x);
        CSSX_K xdu[k] = xdu[k] - V[k] * (x[k] * oors[k]);
        slot(D_PS, x);
        CSSX_K {
            const T wk = x[k] * oors[k];
            xds[k] = xds[k] - V[k] * wk;
            xdv[k] = xdv[k] - c.gamm1 * t[k] * wk;
        }
        if constexpr (MAG) {
            slot(D_PBT, x);
            CSSX_K {
                const T wk = x[k] * (T(kOneOver4Pi) * (T(1) / Rho[k]) * oors[k]);
                xdv[k] = xdv[k] - Bt[k] * wk;
                xdw[k] = xdw[k] + Bp[k] * wk;
            }
            slot(D_PBR, x);
            CSSX_K {
                const T wk = x[k] * (T(kOneOver4Pi) * (T(1) / Rho[k]) * oors[k]);
                xdv[k] = xdv[k] - Br[k] * wk;
                xdu[k] = xdu[k] + Bp[k] * wk;
            }
        }
    }
    // ---- Radial_Terms (rhs_mpi.f90:1297-1518); r derivatives already carry dx/dr
    slot(D_RW, x);
    CSSX_K xdw[k] = xdw[k] - U[k] * x[k];
    slot(D_RV, x);
    CSSX_K xdv[k] = xdv[k] - U[k] * x[k];
    slot(D_RU, x);
    CSSX_K {
        xdu[k] = xdu[k] - U[k] * x[k];
        xdrho[k] = xdrho[k] - Rho[k] * x[k];
    }
    slot(D_RS, x);
    if constexpr (FL) {
        CSSX_K {
            xdu[k] = xdu[k] - c.gamm1 * (t[k] * x[k] + tbar * tb[k] * dsb);
            xds[k] = xds[k] - U[k] * (x[k] + dsb);
        }
    } else {
        CSSX_K {
            xdu[k] = xdu[k] - c.gamm1 * t[k] * x[k];
            xds[k] = xds[k] - U[k] * x[k];
        }
    }
    if constexpr (MAG) {
        slot(D_RBT, x);
        CSSX_K {
            const T wk = x[k] * ((T(1) / Rho[k]) * T(kOneOver4Pi));
            xdu[k] = xdu[k] - Bt[k] * wk;
            xdw[k] = xdw[k] + Br[k] * wk;
        }
        slot(D_RBP, x);
        CSSX_K {
            const T wk = x[k] * ((T(1) / Rho[k]) * T(kOneOver4Pi));
            xdv[k] = xdv[k] + Br[k] * wk;
            xdu[k] = xdu[k] - Bp[k] * wk;
        }
    }
    T drr[MR];
    field(dr_rho, drr);
    // The r sweep of the density took zero wall derivatives, so that it runs with the other sweeps; theirs enter here,
    // within their reach from the wall (48x96x96 FP32: one launch of 6.9 us less).
    auto wall_part = [&](T e, const T *p) {
        if (e != T(0)) {
            run_load<T, MR, REM != 0>(p, ip0 * (unsigned)n + at, (long)c.nphi * n, x);
            CSSX_K drr[k] = drr[k] + e * x[k];
        }
    };
    wall_part(erl, H.rr_lo);
    wall_part(erh, H.rr_hi);
    // ---- Density_Terms_Theta: the wall derivatives that zero the normal momentum tendency
    //      (rhs_mpi.f90:1553-1564), from the end points' own lanes
    {
        const T rvp = rv * c.invpconst;
        const T wl = rvp * xdw[0] * Rho[0] / t[0];
        T e[MR];
        CSSX_K e[k] = xdw[k];
        const T we = G.pick(e, G.m - 1);
        CSSX_K e[k] = Rho[k];
        const T re = G.pick(e, G.m - 1);
        CSSX_K e[k] = t[k];
        const T hv = rvp * we * re / G.pick(e, G.m - 1);
        const T hn = from_next(G.last ? hv : T(0));   // row n-1 alone in its lane: passed to row n-2's
        dth(6, rs, H.brho, G.first ? wl : T(0), G.at_n2 ? (G.jn2 == nl - 1 ? hv : hn) : T(0), x);
        CSSX_K {
            T wk = ri * x[k];
            xdrho[k] = xdrho[k] - W[k] * wk;
            wk = wk * (T(1) / Rho[k]);
            xdw[k] = xdw[k] - c.pconst * wk * t[k];
        }
    }
    // ---- Density_Terms_Radial
    if constexpr (FL) {
        CSSX_K {
            xdu[k] = xdu[k] - c.pconst * ((t[k] * (T(1) / Rho[k])) * drr[k] + tr * ta[k] * drb);
            xdrho[k] = xdrho[k] - U[k] * (drr[k] + drb);
        }
    } else {
        CSSX_K {
            xdrho[k] = xdrho[k] - U[k] * drr[k];
            xdu[k] = xdu[k] - c.pconst * t[k] * (drr[k] * (T(1) / Rho[k]));
        }
    }
    if (c.top_relax && ir == c.nr - 1) {
        const T dt_ = c.damp * (c.gamma - T(2));
        CSSX_K {
            const T dT = FL ? c.dT0top - tbar * tb[k] : c.T0 - t[k];
            xdrho[k] = xdrho[k] + Rho[k] * dT / (dt_ * t[k]);
            xds[k] = xds[k] - c.Cv * dT / (dt_ * t[k]);
        }
    }
    if (c.xi_on) { CSSX_K xdrho[k] = c.xi2 * xdrho[k]; }
    auto closure = [&](int iv, T(&v)[MR]) {   // learned closure tendency
        if (!ext) return;
        float e[MR];
        run_load<float, MR, CHK>(ext + ((long)iv * N + base), at, N - base, e);
        CSSX_K v[k] += (T)e[k];
    };
    closure(0, xdrho);
    closure(1, xdw);
    closure(2, xdv);
    closure(3, xdu);
    closure(4, xds);
    // induction: u x B
    auto induct = [&](int q, T(&v)[MR]) {
        CSSX_K v[k] = q == 0 ? V[k] * Br[k] - U[k] * Bp[k] : q == 1 ? U[k] * Bt[k] - W[k] * Br[k] : W[k] * Bp[k] - V[k] * Bt[k];
        closure(5 + q, v);
    };
    if (!active) return;
    if (F.stage == 0) {
        auto put = [&](int iv, const T(&v)[MR]) { line_store<T, MR>(dv + ((long)iv * N + base), at, G, v); };
        put(0, xdrho);
        put(1, xdw);
        put(2, xdv);
        put(3, xdu);
        put(4, xds);
        if constexpr (MAG) {
#pragma unroll
            for (int q = 0; q < 3; q++) {
                induct(q, x);
                put(5 + q, x);
            }
        }
        return;
    }
    // st may alias F.y1 (the stage state is updated in place): this workgroup alone reads and writes its
    // pencils, and every read of st happened above
    constexpr int NV = MAG ? 8 : 5;
    auto run = [&](auto &R, int iv, const T(&v)[MR]) { R.finish(F, c, G, iv, base, at, it0, ir, v); };
    auto rest = [&](auto &R) {
        if constexpr (MAG) {
#pragma unroll
            for (int q = 0; q < 3; q++) {
                induct(q, x);
                run(R, 5 + q, x);
            }
        }
    };
    auto plain = [&](auto &R) {
        R.load(F, N, base, at);
        run(R, 0, xdrho);
        run(R, 1, xdw);
        run(R, 2, xdv);
        run(R, 3, xdu);
        run(R, 4, xds);
        rest(R);
    };
    if (F.stage == 1) {
        StageRun<T, MR, NV, 1, CHK> R;
        R.load(F, N, base, at);
        if (F.dif && F.corr) {
            // the SLD march left rho..s uncorrected: viscous heating, then mass diffusion (final_point)
            auto vel = [&](int iv, const T(&u)[MR]) {
                CSSX_K {
                    if (F.visc) R.s[4][k] = R.s[4][k] - u[k] * R.s[iv][k] * (T(1) / t[k]);
                    if (F.mass) R.s[iv][k] = R.s[iv][k] - (T(1) / Rho[k]) * u[k] * R.s[0][k];
                }
            };
            vel(1, W);
            vel(2, V);
            vel(3, U);
            if (F.mass) { CSSX_K R.s[4][k] = R.s[4][k] - F.gcv * (T(1) / Rho[k]) * R.s[0][k]; }
        }
        if constexpr (MAG) {
            if (F.dif && F.ohm) {   // SLD Ohmic heating (k_sld_finish's operations in their order)
                auto take = [&](int q, const T(&b)[MR]) {
                    T C[MR];
                    field(F.ohm + (long)q * N, C);
                    CSSX_K R.s[4][k] = R.s[4][k] - b[k] * C[k] * (T(0.5 * kOneOver4Pi) * (T(1) / Rho[k]) * (T(1) / t[k]));
                };
                take(0, Bt);
                take(1, Bp);
                take(2, Br);
            }
        }
        run(R, 0, xdrho);
        run(R, 1, xdw);
        run(R, 2, xdv);
        run(R, 3, xdu);
        run(R, 4, xds);
        rest(R);
    } else if (F.stage == 4) {
        StageRun<T, MR, NV, 4, CHK> R;
        plain(R);
    } else {
        StageRun<T, MR, NV, 2, CHK> R;
        plain(R);
    }
#undef CSSX_K
}

template <typename T, int MR, int REM, bool MAG, bool CUT>
__global__ __launch_bounds__(256, (MR * sizeof(T) > 16 ? 1 : 2)) void k_rhs_line(Consts<T> c, Prof<T> P, const T *st, const T *B, const T *dr_rho, T *dv,
                                                     StageFuse<T> F, const float *__restrict__ ext, const T *D,
                                                     LineTheta<T> H) {
    __shared__ LineCut<T, 7, 4> cut;
    // the last workgroup's last lane may reach past the fields' end
    if (REM != 0 && blockIdx.x == gridDim.x - 1 && blockIdx.y == gridDim.y - 1)
        rhs_line<T, MR, REM, MAG, CUT, true>(c, P, st, B, dr_rho, dv, F, ext, D, H, cut);
    else
        rhs_line<T, MR, REM, MAG, CUT, false>(c, P, st, B, dr_rho, dv, F, ext, D, H, cut);
}

}  // namespace cssx
