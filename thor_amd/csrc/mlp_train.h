// Training kernels of the per-column MLP for the fused network shape (256
// hidden units, n_in <= 128, n_out <= 64): one mini-batch is two launches.
//
// k_train_rows runs forward and backward for 32 rows per block with the
// activations in LDS and the pre-activations in registers; k_train_weights
// forms the weight gradients from what it left, applies Adam and refreshes the
// BF16 operand copies. The layer-by-layer form (k_gemm, k_mse, k_gelu_back,
// k_colsum, k_adam, the copies: 24 launches and a host wait per batch) took
// 361 us per batch of 512 at 81 -> 256 -> 256 -> 40, 212 of them in five
// gradient products of 8 to 16 blocks that walked K 32 at a time through
// element-wise staging; a batch is 0.33 GFLOP, so it is bound by the chain of
// its launches and of the layers inside them, not by the matrix cores: 17 + 6 us
// here (an epoch of 16 384 rows 11.6 -> 0.89 ms, its shuffle and the parameters'
// copy back included).
//
// Operands of the gradient products are kept as fragments: for 32 rows b and a
// tile of 16 units mt, lane l's eight values (rows 8 (l / 16) + e, unit
// l % 16) are 16 contiguous bytes at ((b MT + mt) 64 + l) 8, so that
// dW = A^T dZ reads both operands with one load per lane and 32 rows.
#pragma once
#include "mlp_kernels.h"

namespace thor {
namespace mlp {

struct TrainArgs {
    const float *X, *Y;  // [n][nin], [n][nout]
    const int *idx;      // rows of the batch (null: 0 .. rows - 1)
    long rows;
    InferWeights w;              // forward operands
    const uint16_t *wa2, *wa3;   // W2 [256 x 256], W3 [256 x 64] as A operands (rows = inputs of the layer)
    float scale;                 // 2 / (rows n_out)
    uint16_t *fX, *fH1, *fH2, *fZ1, *fZ2, *fY;  // fragments of the inputs, activations and deltas
    float *bpart;                // [blocks][256 + 256 + 64] bias-gradient sums of each block
    double *part;                // [blocks] sums of squared errors
};
constexpr int kBiasCols = 256 + 256 + 64;

// Fragments of MT 16-unit tiles of an LDS array [32 rows][ld].
__device__ __forceinline__ void write_frags(const uint16_t *s, int ld, int MT, uint16_t *dst) {
    for (int i = threadIdx.x; i < MT * 64; i += kInferThreads) {
        const int mt = i >> 6, l = i & 63, u = 16 * mt + (l & 15), r = 8 * (l >> 4);
        v8s v;
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = (short)s[(r + e) * ld + u];
        *(v8s *)&dst[((size_t)blockIdx.x * MT * 64 + i) * 8] = v;
    }
}

// acc[ti][tj] += W-operand tiles (stored by k_frag_bf16 order, read from
// memory) times the LDS activations, as layer_regs.
template <int NT, int KT>
__device__ __forceinline__ void layer_mem(const uint16_t *sX, int ldx, const uint16_t *Wt, int nt0, int lane,
                                          v4f acc[2][NT]) {
    v8s w[NT][KT];
#pragma unroll
    for (int tj = 0; tj < NT; tj++)
#pragma unroll
        for (int kt = 0; kt < KT; kt++) w[tj][kt] = frag(Wt, KT, nt0 + tj, kt, lane);
    layer_regs<2, NT, KT>(sX, ldx, w, acc);
}

// The lane's sum over the block's 32 samples of each of its four units.
__device__ __forceinline__ void bias_sums(const float d0[4], const float d1[4], float *out) {
    const int li = threadIdx.x & 15;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        float s = d0[e] + d1[e];
#pragma unroll
        for (int m = 1; m < 16; m <<= 1) s += __shfl_xor(s, m);
        if (li == 0) out[e] = s;
    }
}

// Forward and backward of 32 rows: mlp3_rows' products, roundings and
// epilogues (the hidden units 32 w .. of wave w, transposed), then
// dY = scale (Y - T), dZ2 = (dY W3^T) gelu'(Z2), dZ1 = (dZ2 W2^T) gelu'(Z1).
// Z1 and Z2 stay in the registers of the lanes that need them again.
template <int KT1> __global__ __launch_bounds__(kInferThreads, 1) void k_train_rows(TrainArgs g) {
    constexpr int LDH = 256 + 8, LDY = 64 + 8;
    __shared__ __align__(16) uint16_t sX[32 * (32 * KT1 + 8)], sB[32 * LDH], sC[32 * LDH], sD[32 * LDY];
    __shared__ double red[4];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, lq = (lane >> 4) * 4;
    const int nin = g.w.nin, nout = g.w.nout;
    constexpr int kpad = 32 * KT1, ldx = kpad + 8;
    const long r0 = (long)blockIdx.x * 32;
    {
        const int r = tid >> 4, part = tid & 15, kper = kpad / 16;
        const bool rv = r0 + r < g.rows;
        const long src = rv ? (g.idx ? (long)g.idx[r0 + r] : r0 + r) : 0;
#pragma unroll
        for (int j = 0; j < kper; j++) {
            const int k = part * kper + j;
            sX[r * ldx + k] = rv && k < nin ? f2bf_dev(g.X[src * nin + k]) : (uint16_t)0;
        }
    }
    __syncthreads();
    v4f z1[2][2], z2[2][2];
    float b1[2][4], b2[2][4];
#pragma unroll
    for (int tj = 0; tj < 2; tj++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            b1[tj][e] = g.w.b1[32 * wave + 16 * tj + lq + e];
            b2[tj][e] = g.w.b2[32 * wave + 16 * tj + lq + e];
        }
    layer_mem<2, KT1>(sX, ldx, g.w.W1t, 2 * wave, lane, z1);
    write_frags(sX, ldx, 2 * KT1, g.fX);
#pragma unroll
    for (int ti = 0; ti < 2; ti++)
#pragma unroll
        for (int tj = 0; tj < 2; tj++)
            store_gelu4(sB, LDH, 16 * ti + li, 32 * wave + 16 * tj + lq, z1[ti][tj], b1[tj]);
    __syncthreads();
    layer_mem<2, 8>(sB, LDH, g.w.W2t, 2 * wave, lane, z2);
    write_frags(sB, LDH, 16, g.fH1);
#pragma unroll
    for (int ti = 0; ti < 2; ti++)
#pragma unroll
        for (int tj = 0; tj < 2; tj++)
            store_gelu4(sC, LDH, 16 * ti + li, 32 * wave + 16 * tj + lq, z2[ti][tj], b2[tj]);
    __syncthreads();
    if (wave < 4) {
        v4f y[2][1];
        layer_mem<1, 8>(sC, LDH, g.w.W3t, wave, lane, y);
        float d[2][4];
        double sq = 0.0;
#pragma unroll
        for (int ti = 0; ti < 2; ti++) {
            const long r = r0 + 16 * ti + li;
            const bool rv = r < g.rows;
            const long src = rv ? (g.idx ? (long)g.idx[r] : r) : 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int col = 16 * wave + lq + e;
                float diff = 0.f;
                if (rv && col < nout) diff = y[ti][0][e] + g.w.b3[col] - g.Y[src * nout + col];
                sq += (double)diff * diff;
                d[ti][e] = g.scale * diff;
            }
            *(uint2 *)&sD[(16 * ti + li) * LDY + 16 * wave + lq] =
                make_uint2(f2bf2(d[ti][0], d[ti][1]), f2bf2(d[ti][2], d[ti][3]));
        }
        bias_sums(d[0], d[1], g.bpart + (size_t)blockIdx.x * kBiasCols + 512 + 16 * wave + lq);
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) sq += __shfl_xor(sq, m);
        if (lane == 0) red[wave] = sq;
    }
    write_frags(sC, LDH, 16, g.fH2);
    __syncthreads();
    if (tid == 0) g.part[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
    // deltas of a hidden layer: acc = dH, then d = dH gelu'(z + b), kept as BF16
    auto delta = [&](const v4f (&dh)[2][2], const v4f (&z)[2][2], const float (&b)[2][4], uint16_t *s, float *bp) {
#pragma unroll
        for (int tj = 0; tj < 2; tj++) {
            float d[2][4];
            const int u = 32 * wave + 16 * tj + lq;
#pragma unroll
            for (int ti = 0; ti < 2; ti++) {
#pragma unroll
                for (int e = 0; e < 4; e++) d[ti][e] = dh[ti][tj][e] * gelu_grad(z[ti][tj][e] + b[tj][e]);
                *(uint2 *)&s[(16 * ti + li) * LDH + u] = make_uint2(f2bf2(d[ti][0], d[ti][1]), f2bf2(d[ti][2], d[ti][3]));
            }
            bias_sums(d[0], d[1], bp + u);
        }
    };
    v4f dh[2][2];
    layer_mem<2, 2>(sD, LDY, g.wa3, 2 * wave, lane, dh);
    write_frags(sD, LDY, 4, g.fY);
    delta(dh, z2, b2, sB, g.bpart + (size_t)blockIdx.x * kBiasCols + 256);  // sB: H1 was read before the last barriers
    __syncthreads();
    layer_mem<2, 8>(sB, LDH, g.wa2, 2 * wave, lane, dh);
    write_frags(sB, LDH, 16, g.fZ2);
    delta(dh, z1, b1, sC, g.bpart + (size_t)blockIdx.x * kBiasCols);  // sC: H2 was read before the last barriers
    __syncthreads();
    write_frags(sC, LDH, 16, g.fZ1);
}

struct AdamArgs {
    float *w, *m, *v;  // null m: gradients only
    float lr, b1, b2, eps, bc1, bc2;
};
__device__ __forceinline__ float adam_step(const AdamArgs &a, long i, float g) {
    const float m = a.b1 * a.m[i] + (1.f - a.b1) * g;
    const float v = a.b2 * a.v[i] + (1.f - a.b2) * g * g;
    a.m[i] = m;
    a.v[i] = v;
    const float w = a.w[i] - a.lr * (m / a.bc1) / (sqrtf(v / a.bc2) + a.eps);
    a.w[i] = w;
    return w;
}

struct GradArgs {
    const uint16_t *fX, *fH1, *fH2, *fZ1, *fZ2, *fY;
    const float *bpart;
    int nblk, nin, nout, kpad;  // nblk: 32-row groups
    float *grad;                // flat gradients (null while training)
    AdamArgs adam;
    uint16_t *wt1, *wt2, *wt3, *wa2, *wa3;  // BF16 operand copies to refresh (training)
};

// Weight gradients, 32 x 32 entries per 4-wave block: the waves take every
// fourth group of 32 rows, their partial tiles are added in wave order in LDS,
// and each thread finishes four entries: the gradient, or Adam's update and
// the entry's BF16 copies in operand order. Blocks past the tiles sum the
// biases' partial sums, 64 columns each.
__global__ __launch_bounds__(256) void k_train_weights(GradArgs g) {
    __shared__ float s[4][32 * 33];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const long ob1 = (long)g.nin * 256, oW2 = ob1 + 256, ob2 = oW2 + 65536, oW3 = ob2 + 256, ob3 = oW3 + 256L * g.nout;
    const int t1 = (g.nin + 31) / 32 * 8, t3 = 8 * ((g.nout + 31) / 32);
    int b = blockIdx.x;
    if (b >= t1 + 64 + t3) {  // biases: 64 of the 576 columns
        float *q = &s[0][0];
        const int col = (b - (t1 + 64 + t3)) * 64 + lane;
        float sum = 0.f;
        for (int k = wave; k < g.nblk; k += 4) sum += g.bpart[(size_t)k * kBiasCols + col];
        q[wave * 64 + lane] = sum;
        __syncthreads();
        if (wave) return;
        sum = q[lane] + q[64 + lane] + q[128 + lane] + q[192 + lane];
        const long i = col < 256 ? ob1 + col : col < 512 ? ob2 + col - 256 : ob3 + col - 512;
        if (col >= 512 + g.nout) return;
        if (g.adam.m) adam_step(g.adam, i, sum);
        else g.grad[i] = sum;
        return;
    }
    const uint16_t *fa, *fb;
    int MA, MB, i0, n0, K, N, layer;  // tiles per group of both operands; first row and column; size
    if (b < t1) layer = 1, fa = g.fX, fb = g.fZ1, MA = g.kpad / 16, MB = 16, i0 = b / 8 * 32, n0 = b % 8 * 32, K = g.nin, N = 256;
    else if ((b -= t1) < 64) layer = 2, fa = g.fH1, fb = g.fZ2, MA = 16, MB = 16, i0 = b / 8 * 32, n0 = b % 8 * 32, K = 256, N = 256;
    else b -= 64, layer = 3, fa = g.fH2, fb = g.fY, MA = 16, MB = 4, i0 = b % 8 * 32, n0 = b / 8 * 32, K = 256, N = g.nout;
    v4f acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
        for (int y = 0; y < 2; y++) acc[x][y] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int k0 = wave; k0 < g.nblk; k0 += 16) {  // four groups' operands in flight
        v8s a[4][2], c[4][2];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int k = min(k0 + 4 * q, g.nblk - 1);
#pragma unroll
            for (int t = 0; t < 2; t++) {
                a[q][t] = *(const v8s *)&fa[(((size_t)k * MA + i0 / 16 + t) * 64 + lane) * 8];
                c[q][t] = *(const v8s *)&fb[(((size_t)k * MB + n0 / 16 + t) * 64 + lane) * 8];
            }
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
            if (k0 + 4 * q >= g.nblk) break;
#pragma unroll
            for (int x = 0; x < 2; x++)
#pragma unroll
                for (int y = 0; y < 2; y++) acc[x][y] = mfma32(a[q][x], c[q][y], acc[x][y]);
        }
    }
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
        for (int y = 0; y < 2; y++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                s[wave][(16 * x + (lane >> 4) * 4 + e) * 33 + 16 * y + (lane & 15)] = acc[x][y][e];
    __syncthreads();
    const long ow = layer == 1 ? 0 : layer == 2 ? oW2 : oW3;
    for (int j = 0; j < 4; j++) {
        const int x = (tid >> 5) + 8 * j, y = tid & 31, i = i0 + x, n = n0 + y;
        if (i >= K || n >= N) continue;
        const float gr = s[0][x * 33 + y] + s[1][x * 33 + y] + s[2][x * 33 + y] + s[3][x * 33 + y];
        const long at = ow + (long)i * N + n;
        if (!g.adam.m) {
            g.grad[at] = gr;
            continue;
        }
        const uint16_t h = f2bf_dev(adam_step(g.adam, at, gr));
        // operand order of W (k = i) and of W as the A operand (rows i, k = n)
        auto put = [&](uint16_t *d, int KT, int row, int k) {
            d[(((size_t)(row >> 4) * KT + (k >> 5)) * 64 + (row & 15) + 16 * ((k & 31) >> 3)) * 8 + (k & 7)] = h;
        };
        if (layer == 1) put(g.wt1, g.kpad / 32, n, i);
        else if (layer == 2) put(g.wt2, 8, n, i), put(g.wa2, 8, i, n);
        else put(g.wt3, 8, n, i), put(g.wa3, 2, i, n);
    }
}

} // namespace mlp
} // namespace thor
