// Loss gradient and Adam step of the 216-128-128-8 network in three launches (gfx950).  Included by
// cssx_closure.hip after the activation functions.
//
//   k_train_rows   one workgroup per 32 rows: forward, loss, and the backward pass to dZ1 with the
//                  activations in LDS and registers.  A wavefront owns 16 of the 128 units; the weights it
//                  needs for all five products are 17 16-byte loads per lane, issued at the start.  It leaves
//                  X, H1, H2, dY, dZ2 and dZ1 transposed in memory (an accumulator holds four consecutive
//                  rows of one unit: an 8-byte store), because the weight gradients sum over rows.
//   k_train_wgrad  dW = A^T B over the rows: both operands are contiguous along the summed index, so a
//                  fragment is one 16-byte load; wavefront tiles of 32 x 32, the rows split over workgroups,
//                  each writing its partial sum.
//   k_train_apply  sums the partials (and the bias gradients' and the loss'), and with ADAM updates the
//                  weights and their BF16 copies, natural and transposed.
//
// The rounding points are those of the layer-by-layer path (BF16 activations and deltas, FP32 accumulation
// in the same K order, FP32 bias sums); the partial sums are added in a fixed order, without atomics.
// Bound by launch and memory latency: a step on 8192 rows moves 14 MB and does 1.8 GFLOP in 16 + 12 + 5 us
// (the row kernel is one load -> seven dependent phases per workgroup).  Layer by layer it took 14 launches
// and about 400 us (three column sums of 98 us each, whose lanes walked 512 rows one after another, and eight
// products of 14 us in 32 x 32 tiles with strided operand loads).
#pragma once

namespace cssx {

constexpr int kTrH = 128, kTrRows = 32;          // hidden width, rows per workgroup
constexpr int kTrK1 = 224;                       // 216 features padded to 7 K steps of 32
constexpr int kTrXs = 232, kTrHs = 136;          // LDS row strides (BF16): an odd number of 16-byte units
constexpr int kTrBias = 2 * kTrH + kOut;         // bias gradients per workgroup: b1, b2, b3
constexpr int kTrSplit = 32;                     // most row splits of the weight gradients
constexpr int kTrWT = kTrH * kTrK1 + kTrH * kTrH + 16 * kTrH;   // transposed weights: W1T, W2T, W3T (16 rows)
constexpr int kTrWaveTiles = 28 + 16 + 4;        // 32 x 32 tiles of dW1 (216 x 128), dW2 (128 x 128), dW3 (128 x 8)

typedef __bf16 cssx_bf16x4 __attribute__((ext_vector_type(4)));

struct TrainBufs {
    cssx_bf16 *XT, *H1T, *H2T, *dYT, *dZ2T, *dZ1T;   // [unit][row], ld rows apart
    long ld;
    float *bias, *loss;                              // per workgroup: kTrBias sums, squared error
};

__global__ __launch_bounds__(512) void k_train_rows(const cssx_bf16 *__restrict__ X, const float *__restrict__ Tg, int rows,
                                                    const cssx_bf16 *__restrict__ WT, const cssx_bf16 *__restrict__ W2,
                                                    const cssx_bf16 *__restrict__ W3, const float *__restrict__ b1,
                                                    const float *__restrict__ b2, const float *__restrict__ b3, TrainBufs o) {
    __shared__ __align__(16) cssx_bf16 Xs[kTrRows * kTrXs], H1s[kTrRows * kTrHs], H2s[kTrRows * kTrHs], dYs[kTrRows * kOut];
    __shared__ float sh3[2][kOut + 1];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, kg = lane >> 4, c = 16 * w + li;
    const int r0 = blockIdx.x * kTrRows;
    const cssx_bf16 zero = (cssx_bf16)0.0f;
    const cssx_bf16x8 z8 = {zero, zero, zero, zero, zero, zero, zero, zero};
    // ---- this wavefront's weights: unit c's rows of W1T, W2T, W2 and W3, W3T's row li
    cssx_bf16x8 f1[7], f2[4], f3[4], g2[4], g3;
#pragma unroll
    for (int s = 0; s < 7; s++) f1[s] = *(const cssx_bf16x8 *)(WT + (long)c * kTrK1 + s * 32 + kg * 8);
    const cssx_bf16 *W2T = WT + kTrH * kTrK1, *W3T = W2T + kTrH * kTrH;
#pragma unroll
    for (int s = 0; s < 4; s++) {
        f2[s] = *(const cssx_bf16x8 *)(W2T + (long)c * kTrH + s * 32 + kg * 8);
        f3[s] = *(const cssx_bf16x8 *)(W3T + (long)li * kTrH + s * 32 + kg * 8);
        g2[s] = *(const cssx_bf16x8 *)(W2 + (long)c * kTrH + s * 32 + kg * 8);
    }
    g3 = kg == 0 ? *(const cssx_bf16x8 *)(W3 + (long)c * kOut) : z8;
    const float bb1 = b1[c], bb2 = b2[c], bb3 = li < kOut ? b3[li] : 0.0f;
    // ---- X tile, rows past the batch and the K padding zero
    for (int t = tid; t < kTrRows * (kTrXs / 8); t += 512) {
        const int r = t / (kTrXs / 8), q = t - r * (kTrXs / 8);
        *(cssx_bf16x8 *)(Xs + r * kTrXs + q * 8) =
            (r0 + r < rows && q < kFeat / 8) ? *(const cssx_bf16x8 *)(X + (long)(r0 + r) * kFeat + q * 8) : z8;
    }
    __syncthreads();
    // ---- layer 1
    float Z1[2][4], Z2[2][4];
    auto put = [&](cssx_bf16 *S, cssx_bf16 *Tm, int rb, const cssx_bf16x4 &h) {
        // four consecutive rows of unit c: into the LDS rows and the transposed copy
#pragma unroll
        for (int r = 0; r < 4; r++) S[(rb * 16 + kg * 4 + r) * kTrHs + c] = h[r];
        *(cssx_bf16x4 *)(Tm + (long)c * o.ld + r0 + rb * 16 + kg * 4) = h;
    };
#pragma unroll
    for (int rb = 0; rb < 2; rb++) {
        cssx_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 7; s++)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const cssx_bf16x8 *)(Xs + (rb * 16 + li) * kTrXs + s * 32 + kg * 8),
                                                          f1[s], acc, 0, 0, 0);
        cssx_bf16x4 h;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            Z1[rb][r] = acc[r] + bb1;
            h[r] = (cssx_bf16)gelu(Z1[rb][r]);
        }
        put(H1s, o.H1T, rb, h);
    }
    // X transposed: 8 rows of one feature per task
    for (int t = tid; t < kFeat * 4; t += 512) {
        const int q = t >> 2, ch = t & 3;
        cssx_bf16x8 v;
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = Xs[(ch * 8 + e) * kTrXs + q];
        *(cssx_bf16x8 *)(o.XT + (long)q * o.ld + r0 + ch * 8) = v;
    }
    __syncthreads();
    // ---- layer 2
#pragma unroll
    for (int rb = 0; rb < 2; rb++) {
        cssx_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 4; s++)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const cssx_bf16x8 *)(H1s + (rb * 16 + li) * kTrHs + s * 32 + kg * 8),
                                                          f2[s], acc, 0, 0, 0);
        cssx_bf16x4 h;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            Z2[rb][r] = acc[r] + bb2;
            h[r] = (cssx_bf16)gelu(Z2[rb][r]);
        }
        put(H2s, o.H2T, rb, h);
    }
    __syncthreads();
    // ---- layer 3, loss and its gradient: wavefronts 0 and 1, 16 rows each
    if (w < 2) {
        cssx_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 4; s++)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const cssx_bf16x8 *)(H2s + (w * 16 + li) * kTrHs + s * 32 + kg * 8),
                                                          f3[s], acc, 0, 0, 0);
        float d2 = 0.f, sg = 0.f;
        cssx_bf16x4 gb;
        const float n = (float)((long)rows * kOut);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = r0 + w * 16 + kg * 4 + r;
            const bool ok = row < rows && li < kOut;
            const float d = ok ? (acc[r] + bb3) - Tg[(long)row * kOut + li] : 0.0f;
            const float g = 2.0f * d / n;
            gb[r] = (cssx_bf16)g;
            sg += g;
            d2 += d * d;
            if (li < kOut) dYs[(w * 16 + kg * 4 + r) * kOut + li] = gb[r];
        }
        if (li < kOut) *(cssx_bf16x4 *)(o.dYT + (long)li * o.ld + r0 + w * 16 + kg * 4) = gb;
        sg += __shfl_xor(sg, 16, 64);
        sg += __shfl_xor(sg, 32, 64);
        for (int s = 32; s > 0; s >>= 1) d2 += __shfl_xor(d2, s, 64);
        if (lane < kOut) sh3[w][lane] = sg;
        if (lane == 0) sh3[w][kOut] = d2;
    }
    __syncthreads();
    float *bias = o.bias + (long)blockIdx.x * kTrBias;
    if (tid < kOut) bias[2 * kTrH + tid] = sh3[0][tid] + sh3[1][tid];
    if (tid == kOut) o.loss[blockIdx.x] = sh3[0][kOut] + sh3[1][kOut];
    // ---- dZ2 = (dY W3^T) GELU'(Z2), into H1's LDS rows (layer 2 is done with them)
    float s2 = 0.f, s1 = 0.f;
#pragma unroll
    for (int rb = 0; rb < 2; rb++) {
        cssx_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        const cssx_bf16x8 a = kg == 0 ? *(const cssx_bf16x8 *)(dYs + (rb * 16 + li) * kOut) : z8;
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, g3, acc, 0, 0, 0);
        cssx_bf16x4 h;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float d = acc[r] * gelu_grad(Z2[rb][r]);
            s2 += d;
            h[r] = (cssx_bf16)d;
        }
        put(H1s, o.dZ2T, rb, h);
    }
    __syncthreads();
    // ---- dZ1 = (dZ2 W2^T) GELU'(Z1)
#pragma unroll
    for (int rb = 0; rb < 2; rb++) {
        cssx_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 4; s++)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const cssx_bf16x8 *)(H1s + (rb * 16 + li) * kTrHs + s * 32 + kg * 8),
                                                          g2[s], acc, 0, 0, 0);
        cssx_bf16x4 h;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float d = acc[r] * gelu_grad(Z1[rb][r]);
            s1 += d;
            h[r] = (cssx_bf16)d;
        }
        *(cssx_bf16x4 *)(o.dZ1T + (long)c * o.ld + r0 + rb * 16 + kg * 4) = h;
    }
    s1 += __shfl_xor(s1, 16, 64);
    s1 += __shfl_xor(s1, 32, 64);
    s2 += __shfl_xor(s2, 16, 64);
    s2 += __shfl_xor(s2, 32, 64);
    if (kg == 0) {
        bias[c] = s1;
        bias[kTrH + c] = s2;
    }
}

// partial dW of rows [blockIdx.y*chunk, +chunk) into part + blockIdx.y*np (layout of the parameters)
__global__ __launch_bounds__(256) void k_train_wgrad(TrainBufs o, int rows, int chunk, long oW2, long oW3, long np,
                                                     float *__restrict__ part) {
    const int lane = threadIdx.x & 63, li = lane & 15, kg = lane >> 4;
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
    const cssx_bf16 *A, *B;
    int m0, n0, M, N;
    long off;
    if (t < 28) {
        A = o.XT; B = o.dZ1T; m0 = (t >> 2) * 32; n0 = (t & 3) * 32; M = kFeat; N = kTrH; off = 0;
    } else if (t < 44) {
        A = o.H1T; B = o.dZ2T; m0 = ((t - 28) >> 2) * 32; n0 = ((t - 28) & 3) * 32; M = kTrH; N = kTrH; off = oW2;
    } else {
        A = o.H2T; B = o.dYT; m0 = (t - 44) * 32; n0 = 0; M = kTrH; N = kOut; off = oW3;
    }
    const cssx_bf16 zero = (cssx_bf16)0.0f;
    const cssx_bf16x8 z8 = {zero, zero, zero, zero, zero, zero, zero, zero};
    const int k0 = blockIdx.y * chunk, k1 = min(k0 + chunk, (rows + kTrRows - 1) / kTrRows * kTrRows);
    const cssx_bf16 *a[2], *b[2];
    bool am[2], bm[2];
#pragma unroll
    for (int q = 0; q < 2; q++) {
        am[q] = m0 + q * 16 + li < M;
        bm[q] = n0 + q * 16 + li < N;
        a[q] = A + (long)(am[q] ? m0 + q * 16 + li : 0) * o.ld + kg * 8;
        b[q] = B + (long)(bm[q] ? n0 + q * 16 + li : 0) * o.ld + kg * 8;
    }
    cssx_f32x4 acc[2][2] = {};
    constexpr int D = 4;   // K steps whose loads are in flight together
    for (int kb = k0; kb < k1; kb += 32 * D) {
        cssx_bf16x8 fa[D][2], fb[D][2];
#pragma unroll
        for (int d = 0; d < D; d++) {
            const int k = kb + 32 * d;
#pragma unroll
            for (int q = 0; q < 2; q++) {
                fa[d][q] = k < k1 ? *(const cssx_bf16x8 *)(a[q] + k) : z8;
                fb[d][q] = k < k1 ? *(const cssx_bf16x8 *)(b[q] + k) : z8;
            }
        }
#pragma unroll
        for (int d = 0; d < D; d++)
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[d][i], fb[d][j], acc[i][j], 0, 0, 0);
    }
    float *out = part + (long)blockIdx.y * np + off;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int n = n0 + j * 16 + li;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + i * 16 + kg * 4 + r;
                if (m < M && n < N) out[(long)m * N + n] = acc[i][j][r];
            }
        }
}

struct AdamArgs {
    float *W, *M, *V;
    cssx_bf16 *Wb, *WT;
    float lr, b1, b2, eps, c1, c2;
};

// a weight's BF16 copies: natural, and transposed for the forward products
__device__ __forceinline__ void store_weight(cssx_bf16 *Wb, cssx_bf16 *WT, long i, long oW2, long oW3, float w) {
    const cssx_bf16 v = (cssx_bf16)w;
    Wb[i] = v;
    if (i < (long)kFeat * kTrH) {
        WT[(i % kTrH) * kTrK1 + i / kTrH] = v;
    } else if (i >= oW2 && i < oW2 + (long)kTrH * kTrH) {
        const long j = i - oW2;
        WT[kTrH * kTrK1 + (j % kTrH) * kTrH + j / kTrH] = v;
    } else if (i >= oW3 && i < oW3 + (long)kTrH * kOut) {
        const long j = i - oW3;
        WT[kTrH * kTrK1 + kTrH * kTrH + (j % kOut) * kTrH + j / kOut] = v;
    }
}
// both copies of every weight, and the transposed copy's padding
__global__ __launch_bounds__(256) void k_train_copies(const float *__restrict__ W, long np, long oW2, long oW3,
                                                      cssx_bf16 *__restrict__ Wb, cssx_bf16 *__restrict__ WT) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < np) store_weight(Wb, WT, i, oW2, oW3, W[i]);
    if (i < kTrH * (kTrK1 - kFeat)) WT[(i / (kTrK1 - kFeat)) * kTrK1 + kFeat + i % (kTrK1 - kFeat)] = (cssx_bf16)0.0f;
    if (i < (16 - kOut) * kTrH) WT[kTrH * kTrK1 + kTrH * kTrH + kOut * kTrH + i] = (cssx_bf16)0.0f;
}

// G = the summed partials; ADAM: and the update.  Blocks [0, nw): 256 parameters each (biases left out);
// the blocks after: 32 bias gradients each, then the loss.
template <bool ADAM>
__global__ __launch_bounds__(256) void k_train_apply(const float *__restrict__ part, int splits, long np, long ob1, long oW2,
                                                     long ob2, long oW3, long ob3, const float *__restrict__ bias,
                                                     const float *__restrict__ lossp, int nwg, float n, int nw,
                                                     float *__restrict__ G, float *__restrict__ loss, float *loss_out,
                                                     AdamArgs A) {
    __shared__ float sh[8][33];
    auto update = [&](long i, float g) {
        G[i] = g;
        if constexpr (ADAM) {
            const float m = A.b1 * A.M[i] + (1.0f - A.b1) * g;
            const float v = A.b2 * A.V[i] + (1.0f - A.b2) * g * g;
            A.M[i] = m;
            A.V[i] = v;
            const float w = A.W[i] - A.lr * (m / A.c1) / (sqrtf(v / A.c2) + A.eps);
            A.W[i] = w;
            store_weight(A.Wb, A.WT, i, oW2, oW3, w);
        }
    };
    if ((int)blockIdx.x < nw) {
        const long i = (long)blockIdx.x * 256 + threadIdx.x;
        if (i >= np || (i >= ob1 && i < oW2) || (i >= ob2 && i < oW3) || i >= ob3) return;
        float g = 0.f;
#pragma unroll 8
        for (int s = 0; s < splits; s++) g += part[(long)s * np + i];
        update(i, g);
        return;
    }
    const int q = (int)blockIdx.x - nw, p = threadIdx.x & 31, e = threadIdx.x >> 5;
    const bool is_loss = q * 32 >= kTrBias;
    const int col = q * 32 + p;
    float s = 0.f;
    if (is_loss) {
        for (int b = threadIdx.x; b < nwg; b += 256) s += lossp[b];
    } else if (col < kTrBias) {
#pragma unroll 8
        for (int b = e; b < nwg; b += 8) s += bias[(long)b * kTrBias + col];
    }
    sh[e][p] = s;
    __syncthreads();
    if (e == 0) {
        s = 0.f;
#pragma unroll
        for (int k = 0; k < 8; k++) s += sh[k][p];
        if (is_loss) {
            for (int o = 16; o > 0; o >>= 1) s += __shfl_xor(s, o, 32);
            if (p == 0) {
                *loss = s / n;
                if (loss_out) *loss_out = s / n;
            }
        } else if (col < kTrBias) {
            update(col < kTrH ? ob1 + col : col < 2 * kTrH ? ob2 + col - kTrH : ob3 + col - 2 * kTrH, s);
        }
    }
}

}  // namespace cssx
