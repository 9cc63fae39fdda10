// Compact derivative along the contiguous axis (theta, unit row stride) with walls at both ends, for
// gfx950: the operator of derivatives.f90 Dbydt :1010-1262 and D2bydt2 :1265-1477, solved with the
// constant-coefficient recurrences of cssx_uniform.hpp.
//
// Lane j of a pencil holds rows [j*MR, j*MR + MR) in registers (16-byte loads and stores at any
// 4-byte alignment); a wavefront packs as many whole pencils as fit its 64 lanes.  Stencil halos and the
// segment carries move by DPP wave shifts, so a wavefront needs no LDS, no barrier and no plan table.
// Bound by HBM: one read and one write per point.  At 256x512x1024 in FP32 185 us (5.8 TB/s, the rate
// of a bare copy with 32 bytes per lane) against 262 with plan tables in LDS and cyclic reduction; at the ragged
// 90x151x250 26 against 107 us for the fields of one right-hand side, whose lengths no multiple of 8 kept off
// the vector loads.
#include <hip/hip_runtime.h>

#include "cssx_bufio.hpp"
#include "cssx_line.hpp"

namespace cssx {

template <typename T, int ORDER, int MR, int REM>
__global__ __launch_bounds__(256) void k_deriv_line(const DerivLaunch<T> L, const unsigned inv_nl) {
    const DerivJob<T> &J = L.jobs[blockIdx.y];
    const int n = L.n, nl = L.S;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // lane = pl*nl + j (inv_nl = ceil(2^16 / nl): exact for lane < 64); ppw pencils per wavefront
    const int pl = (int)((unsigned)lane * inv_nl >> 16), j = lane - pl * nl, ppw = L.M;
    const unsigned np = (unsigned)L.na * (unsigned)L.nb, id0 = (blockIdx.x * 4 + wv) * ppw;
    if (id0 >= np) return;
    const unsigned id = id0 + pl;
    const bool active = pl < ppw && id < np;
    // values from the wavefront's first pencil on, and the lane's first row from there
    long at0 = (long)id0 * n, total = (long)np * n - at0, at = active ? (long)(pl * n + j * MR) : 0;
    unsigned a = id, b = 0;
    const bool apart = L.nb > 1 && L.sb != (long)L.na * n;   // planes of pencils not back to back
    if (L.nb > 1 && (apart || J.glo || J.ghi || J.mul_a || J.mul_b)) {
        b = id / (unsigned)L.na;
        a = id - b * (unsigned)L.na;
    }
    if (apart) {
        at0 = 0;
        total = (long)(L.nb - 1) * L.sb + (long)L.na * n;
        at = active ? (long)a * n + (long)b * L.sb + j * MR : 0;
    }
    LineShape<MR, REM> G(n, nl, j, active);
    T v[MR], x[MR];
    line_load<T, MR>(J.in + at0, at, total, G, v);
    T lo_val = T(0), hi_val = T(0);
    if (J.glo || J.ghi) {
        const long gbase = (long)a * J.g_a + (long)b * J.g_b;
        if (G.first && J.glo) lo_val = J.glo[gbase];
        if (G.at_n2 && J.ghi) hi_val = J.ghi[gbase];
    }
    if (J.tap_in && active) {
        if (j == 0) J.tap_in[id] = v[0];
        if (j == nl - 1) J.tap_in[J.tap_side + id] = G.pick(v, G.m - 1);
    }
    if (J.pre) {
        T pv[MR];
        line_load<T, MR>(J.pre, j * MR, n, G, pv);
#pragma unroll
        for (int k = 0; k < MR; k++) v[k] *= pv[k];
    }
    const T xn1 = line_solve<T, ORDER, MR>(G, v, J.bdry, lo_val * J.neu_mul, hi_val * J.neu_mul, J.scale, x);
    line_last<T, MR>(G, xn1, x);
    if (!active) return;
    if (J.post) {
        T pw[MR];
        line_load<T, MR>(J.post, j * MR, n, G, pw);
#pragma unroll
        for (int k = 0; k < MR; k++) x[k] *= pw[k];
    }
    if (J.mul_a || J.mul_b) {
        const T pm = (J.mul_a ? J.mul_a[a] : T(1)) * (J.mul_b ? J.mul_b[b] : T(1));
#pragma unroll
        for (int k = 0; k < MR; k++) x[k] *= pm;
    }
    if (J.beta != T(0)) {
        T old[MR];
        line_load<T, MR>(J.out + at0, at, total, G, old);
#pragma unroll
        for (int k = 0; k < MR; k++) x[k] += J.beta * old[k];
    }
    if (J.tap_out) {
        if (j == 0) J.tap_out[id] = x[0];
        if (j == nl - 1) J.tap_out[J.tap_side + id] = G.pick(x, G.m - 1);
    }
    line_store<T, MR>(J.out + at0, at, G, x);
}

// L.M rows per lane: 8 up to 512 rows, 16 up to 1024 (64 lanes); L.S lanes per pencil
template <typename T>
hipError_t launch_deriv_line(const DerivLaunch<T> &L0, int order, hipStream_t stream) {
    DerivLaunch<T> L = L0;
    const int MR = L.M, nl = L.S;
    if ((MR != 8 && MR != 16) || nl != (L.n + MR - 1) / MR || nl > 64 || L.njobs < 1 || L.njobs > kMaxJobs ||
        L.srow != 1 || L.sa != L.n || (L.nb > 1 && L.sb < (long)L.n * L.na) || (long)L.na * L.nb > 0x7fffff00L)
        return hipErrorInvalidValue;
    const int ppw = 64 / nl;
    L.M = ppw;
    const long waves = ((long)L.na * L.nb + ppw - 1) / ppw;
    const dim3 grid((unsigned)((waves + 3) / 4), L.njobs), block(256);
    const unsigned inv = (65536u + nl - 1) / nl;
#define CSSX_LAUNCH_L(MM, RR)                                                                                      \
    do {                                                                                                           \
        if (order == 1) hipLaunchKernelGGL((k_deriv_line<T, 1, MM, RR>), grid, block, 0, stream, L, inv);          \
        else hipLaunchKernelGGL((k_deriv_line<T, 2, MM, RR>), grid, block, 0, stream, L, inv);                     \
    } while (0)
    // the length's remainder is a template parameter of the 8-row kernel (lengths up to 512): 311x333x411
    // in FP32 73 us against 82 with the places of the last rows found at run time
    if (MR == 8) {
        switch (L.n % 8) {
        case 0: CSSX_LAUNCH_L(8, 0); break;
        case 1: CSSX_LAUNCH_L(8, 1); break;
        case 2: CSSX_LAUNCH_L(8, 2); break;
        case 3: CSSX_LAUNCH_L(8, 3); break;
        case 4: CSSX_LAUNCH_L(8, 4); break;
        case 5: CSSX_LAUNCH_L(8, 5); break;
        case 6: CSSX_LAUNCH_L(8, 6); break;
        default: CSSX_LAUNCH_L(8, 7); break;
        }
    } else if (L.n % 16 == 0) {
        CSSX_LAUNCH_L(16, 0);
    } else {
        CSSX_LAUNCH_L(16, -1);
    }
#undef CSSX_LAUNCH_L
    return hipGetLastError();
}

template hipError_t launch_deriv_line<float>(const DerivLaunch<float> &, int, hipStream_t);
template hipError_t launch_deriv_line<double>(const DerivLaunch<double> &, int, hipStream_t);

}  // namespace cssx
